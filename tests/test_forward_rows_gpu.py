"""The 16-bit forward on launches of few query rows (fwd16_rows_kernel).

Such a launch runs one workgroup per 32 rows of a key/value head's query heads, whose waves take
every eighth (head_dim 256: fourth) 32-key block, and with very few rows also cuts the keys into
chunks that a second kernel merges. Checked against the fp64 oracle on every row where that can go
wrong: one row, rows that end inside a tile, heads packed into one tile, fewer blocks than waves,
a last block and a last chunk of one key, causal rows that end before, inside and after a chunk,
every head_dim.

Bounds: V lies in [-1, 1), so rounding P to the input type moves a row of O by at most the unit
roundoff u, and rounding O by as much again; fp32 sums add less than u / 4. L is a sum of at most
8193 fp32 terms of exact products: its error is well under 2e-5.
"""

from __future__ import annotations

import numpy as np
import pytest

import cuflash_attn
import oracle
from conftest import max_abs
from cuflash_attn import synth

UNIT = {"bfloat16": 2.0 ** -9, "float16": 2.0 ** -11}

# B, H, Hkv, Nq, Nk, D, causal
SHAPES = [
    (1, 8, 2, 61, 1025, 128, True),
    (1, 4, 1, 1, 4097, 128, True),
    (2, 2, 2, 1, 8193, 64, False),
    (1, 2, 2, 129, 577, 64, False),
    (1, 8, 8, 700, 700, 64, True),
    (1, 3, 3, 1057, 1057, 128, True),
    (1, 4, 2, 300, 515, 32, True),
    (2, 6, 2, 33, 3000, 96, True),
    (1, 3, 1, 40, 1300, 256, True),
    (1, 2, 2, 300, 300, 256, False),
    (1, 8, 1, 17, 2048, 128, False),
    (20, 32, 8, 1, 70, 64, False),
    (20, 32, 8, 2, 130, 128, True),
]

# B, H, Hkv, keys, D: grouped-query decodes of short caches, which run the same kernel.
DECODES = [(1, 32, 8, 1000, 128), (3, 12, 2, 1, 128), (2, 32, 1, 33, 64), (5, 8, 4, 1024, 32)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_forward_of_few_rows_matches_the_oracle(torch_gpu, dtype, shape):
    B, H, Hkv, Nq, Nk, D, causal = shape
    q = synth.round_to(synth.uniform(1, (B, H, Nq, D)), dtype)
    k, v = (synth.round_to(synth.uniform(s, (B, Hkv, Nk, D)), dtype) for s in (2, 3))
    scale = 2.0 * D ** -0.5
    print(f"[forward rows] {dtype} {shape}", flush=True)
    o, lse = cuflash_attn.flash_attention_forward_ext(
        *(synth.to_torch(x, dtype) for x in (q, k, v)), scale=scale, causal=causal)
    torch_gpu.cuda.synchronize()
    o_ref, l_ref = oracle.forward(q, *(np.repeat(x, H // Hkv, axis=1) for x in (k, v)), scale,
                                  causal)
    assert max_abs(synth.to_numpy(o), o_ref) <= 2.25 * UNIT[dtype]
    assert max_abs(synth.to_numpy(lse), l_ref) <= 2e-5


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("shape", DECODES, ids=lambda s: "-".join(map(str, s)))
def test_short_grouped_decode_matches_the_oracle(torch_gpu, dtype, shape):
    B, H, Hkv, Nk, D = shape
    q = synth.round_to(synth.uniform(1, (B, H, 1, D)), dtype)
    k, v = (synth.round_to(synth.uniform(s, (B, Hkv, Nk, D)), dtype) for s in (2, 3))
    print(f"[short decode] {dtype} {shape}", flush=True)
    for scale in (2.0 * D ** -0.5, 0.0):
        o, lse = cuflash_attn.flash_attention_decode(
            *(synth.to_torch(x, dtype) for x in (q, k, v)), scale=scale)
        torch_gpu.cuda.synchronize()
        o_ref, l_ref = oracle.forward(q, *(np.repeat(x, H // Hkv, axis=1) for x in (k, v)), scale,
                                      False)
        assert max_abs(synth.to_numpy(o), o_ref) <= 2.25 * UNIT[dtype]
        assert max_abs(synth.to_numpy(lse), l_ref) <= 2e-5
