"""Host code and plans of the library in small C++ programs (tests/cpp), compiled here with hipcc and
run without a GPU: what they check stands in each program's first lines."""

from __future__ import annotations

import os
import subprocess

import build as cuflash_build  # cuflash-attn_amd/build.py


def run_program(name, tmp_path, *args):
    exe = tmp_path / name
    env = {k: v for k, v in os.environ.items() if k != "LD_PRELOAD"}
    subprocess.run(
        [cuflash_build.hipcc(), "-x", "hip", "--offload-arch=gfx950", "-O2", "-std=c++17",
         f"-I{cuflash_build.INCLUDE}", f"-I{cuflash_build.CSRC}",
         os.path.join(cuflash_build.TEST_SRC, name + ".cpp"), "-o", str(exe)],
        check=True, env=env)
    proc = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, env=env,
                          timeout=300)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    return proc.stdout


def test_unknown_capture_status_counts_as_captured(tmp_path):
    run_program("test_capture_status", tmp_path)


def test_balanced_paged_split_stays_in_bounds(tmp_path):
    """Over launches that keep the equal splits, that balance, and that are nearly full."""
    run_program("test_paged_split", tmp_path, 3000, 1)


def test_kernel_rules_take_the_measured_faster_kernel(tmp_path):
    run_program("test_kernel_rules", tmp_path)
