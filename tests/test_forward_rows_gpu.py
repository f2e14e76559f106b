"""The 16-bit forward on launches of few query rows (fwd16_rows_kernel).

Such a launch runs one workgroup per 32 rows of a key/value head's query heads, whose waves take
every eighth (head_dim 256: fourth) 32-key block, and with very few rows also cuts the keys into
chunks that a second kernel merges. Checked against the fp64 oracle on every row where that can go
wrong: one row, rows that end inside a tile, heads packed into one tile, fewer blocks than waves,
a last block and a last chunk of one key, causal rows that end before, inside and after a chunk,
merges with several rows' parts in one workgroup, every head_dim. Each shape names the chunks that
it must run in; the host rule is held to that on the CPU, the launches on the GPU.

Bounds: V lies in [-1, 1), so rounding P to the input type moves a row of O by at most the unit
roundoff u, and rounding O by as much again; fp32 sums add less than u / 4. L is a sum of at most
12289 fp32 terms of exact products: its error is well under 2e-5.
"""

from __future__ import annotations

import contextlib

import numpy as np
import pytest

import cuflash_attn
import oracle
from conftest import max_abs
from cuflash_attn import synth
from test_host_rules import run_program

UNIT = {"bfloat16": 2.0 ** -9, "float16": 2.0 ** -11}

# B, H, Hkv, Nq, Nk, D, causal, chunks
SHAPES = [
    (1, 8, 2, 61, 1025, 128, True, 1),
    (1, 4, 1, 1, 4097, 128, True, 6),
    (2, 2, 2, 1, 8193, 64, False, 11),
    (1, 2, 2, 129, 577, 64, False, 1),
    (1, 8, 8, 700, 700, 64, True, 1),
    (1, 3, 3, 1057, 1057, 128, True, 1),
    (1, 4, 2, 300, 515, 32, True, 1),
    (2, 6, 2, 33, 3000, 96, True, 4),
    (1, 3, 1, 40, 1300, 256, True, 4),
    (1, 2, 2, 300, 300, 256, False, 1),
    (1, 8, 1, 17, 2048, 128, False, 4),
    (20, 32, 8, 1, 70, 64, False, 1),
    (20, 32, 8, 2, 130, 128, True, 1),
    # Causal rows that end before a chunk: whole tiles that skip it, and rows inside a tile.
    (1, 1, 1, 1000, 2100, 128, True, 3),
    (1, 1, 1, 600, 4097, 64, True, 6),
    (1, 2, 2, 700, 1100, 256, True, 3),
    (1, 1, 1, 2001, 2001, 64, True, 3),
    (1, 4, 1, 400, 1500, 256, True, 4),
    # A last chunk of one key that one row sees; merges that share a row over two and four groups.
    (1, 1, 1, 64, 12289, 256, True, 25),
    (1, 2, 1, 40, 12289, 96, True, 17),
    (1, 4, 4, 3, 8193, 128, True, 11),
]


@contextlib.contextmanager
def kernels_of(torch, lib):
    """The labels of the kernels that the library launches inside the block (filled at its end)."""
    launched = set()
    torch.cuda.synchronize()
    lib.profile_report()
    lib.profile_enable(True)
    try:
        yield launched
        torch.cuda.synchronize()
    finally:
        lib.profile_enable(False)
        launched.update(lib.profile_report())


def test_shapes_run_in_the_chunks_that_they_name(tmp_path):
    args = [int(x) for shape in SHAPES for x in shape[:7]]
    got = [tuple(map(int, line.split()))
           for line in run_program("test_kernel_rules", tmp_path, *args).splitlines()]
    assert [n for n, _ in got] == [shape[7] for shape in SHAPES]
    # What the comments of SHAPES say of the last chunks.
    last = [shape[4] - (n - 1) * chunk for shape, (n, chunk) in zip(SHAPES, got)]
    assert 1 in last
    assert sum(shape[6] and n > 1 and shape[4] - shape[3] < (n - 1) * chunk
               for shape, (n, chunk) in zip(SHAPES, got)) >= 6


# B, H, Hkv, keys, D: grouped-query decodes of short caches, which run the same kernel.
DECODES = [(1, 32, 8, 1000, 128), (3, 12, 2, 1, 128), (2, 32, 1, 33, 64), (5, 8, 4, 1024, 32)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_forward_of_few_rows_matches_the_oracle(torch_gpu, lib, dtype, shape):
    B, H, Hkv, Nq, Nk, D, causal, chunks = shape
    q = synth.round_to(synth.uniform(1, (B, H, Nq, D)), dtype)
    k, v = (synth.round_to(synth.uniform(s, (B, Hkv, Nk, D)), dtype) for s in (2, 3))
    scale = 2.0 * D ** -0.5
    print(f"[forward rows] {dtype} {shape}", flush=True)
    tensors = [synth.to_torch(x, dtype) for x in (q, k, v)]
    with kernels_of(torch_gpu, lib) as launched:
        o, lse = cuflash_attn.flash_attention_forward_ext(*tensors, scale=scale, causal=causal)
    assert any(label.startswith("forward_combine") for label in launched) == (chunks > 1), launched
    o_ref, l_ref = oracle.forward(q, *(np.repeat(x, H // Hkv, axis=1) for x in (k, v)), scale,
                                  causal)
    assert max_abs(synth.to_numpy(o), o_ref) <= 2.25 * UNIT[dtype]
    assert max_abs(synth.to_numpy(lse), l_ref) <= 2e-5


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("shape", DECODES, ids=lambda s: "-".join(map(str, s)))
def test_short_grouped_decode_matches_the_oracle(torch_gpu, lib, dtype, shape):
    B, H, Hkv, Nk, D = shape
    q = synth.round_to(synth.uniform(1, (B, H, 1, D)), dtype)
    k, v = (synth.round_to(synth.uniform(s, (B, Hkv, Nk, D)), dtype) for s in (2, 3))
    print(f"[short decode] {dtype} {shape}", flush=True)
    for scale in (2.0 * D ** -0.5, 0.0):
        tensors = [synth.to_torch(x, dtype) for x in (q, k, v)]
        with kernels_of(torch_gpu, lib) as launched:
            o, lse = cuflash_attn.flash_attention_decode(*tensors, scale=scale)
        suffix = {"bfloat16": "bf16", "float16": "f16"}[dtype]
        assert launched == {f"decode_rows_{suffix}_d{D}"}
        o_ref, l_ref = oracle.forward(q, *(np.repeat(x, H // Hkv, axis=1) for x in (k, v)), scale,
                                      False)
        assert max_abs(synth.to_numpy(o), o_ref) <= 2.25 * UNIT[dtype]
        assert max_abs(synth.to_numpy(lse), l_ref) <= 2e-5


# B, H, Hkv, Nq, Nk, D: one chunk and several, with a merge over one and over several groups.
SPECIAL = [(1, 4, 4, 300, 300, 64), (1, 2, 2, 700, 1100, 256), (1, 8, 2, 61, 4097, 128),
           (1, 2, 1, 40, 12289, 96)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("shape", SPECIAL, ids=lambda s: "-".join(map(str, s)))
def test_infinities_and_nan_reach_the_rows_that_see_them_and_no_other(torch_gpu, dtype, shape):
    """A NaN or infinite key makes the rows that see it NaN and leaves the others as they were, bit
    for bit; an infinite value reaches its own column only; a key whose scores are -inf has no
    weight (the oracle without that key); rows whose scores are all -inf are NaN with L = -inf."""
    torch = torch_gpu
    B, H, Hkv, Nq, Nk, D = shape
    scale = D ** -0.5
    q = synth.round_to(np.abs(synth.uniform(1, (B, H, Nq, D))) + 0.25, dtype)
    k, v = (synth.round_to(synth.uniform(s, (B, Hkv, Nk, D)), dtype) for s in (2, 3))
    tq, tk, tv = (synth.to_torch(x, dtype) for x in (q, k, v))
    at = Nk - Nq + Nq // 2  # the key that row Nq // 2 is the first to see

    def run(k, v, causal=True):
        out = cuflash_attn.flash_attention_forward_ext(tq, k, v, scale=scale, causal=causal)
        torch.cuda.synchronize()
        return out

    print(f"[special values] {dtype} {shape}", flush=True)
    clean_o, clean_l = run(tk, tv)
    for value in (float("nan"), float("inf")):
        bad = tk.clone()
        bad[:, :, at] = value
        o, lse = run(bad, tv)
        before, seen = slice(None, Nq // 2), slice(Nq // 2, None)
        assert torch.equal(o[:, :, before], clean_o[:, :, before])
        assert torch.equal(lse[:, :, before], clean_l[:, :, before])
        assert bool(o[:, :, seen].isnan().all())
    bad = tv.clone()
    bad[:, :, at, 5] = float("inf")
    o, lse = run(tk, bad)
    assert torch.equal(lse, clean_l)
    rest = torch.arange(D, device="cuda") != 5
    assert torch.equal(o[..., rest], clean_o[..., rest])
    assert not bool(o[:, :, Nq // 2:, 5].isfinite().any())

    bad = tk.clone()
    bad[:, :, at] = float("-inf")
    o, lse = run(bad, tv, causal=False)
    o_ref, l_ref = oracle.forward(
        q, *(np.repeat(np.delete(x, at, axis=2), H // Hkv, axis=1) for x in (k, v)), scale, False)
    assert max_abs(synth.to_numpy(o), o_ref) <= 2.25 * UNIT[dtype]
    assert max_abs(synth.to_numpy(lse), l_ref) <= 2e-5
    o, lse = run(torch.full_like(tk, float("-inf")), tv)
    assert bool(o.isnan().all()) and bool(torch.isneginf(lse).all())
