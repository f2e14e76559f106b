"""The balanced split of a paged grouped-query decode (BalancedArgs in decode.hip).

A paged decode with automatic splits cuts each sequence into as many segments as its length asks
for, so a sequence can have none, one or many, a last segment can be short, and where the cache is
almost full the equal splits of its capacity are kept. Lengths that do each of these are
checked row by row against the fp64 oracle; the bounds are those of an MFMA decode with V in
[-1, 1): the unit roundoff of P and of O, and 2e-5 for L (fp32 sums of exact products).
"""

from __future__ import annotations

import numpy as np
import pytest

import cuflash_attn
import oracle
from conftest import max_abs
from cuflash_attn import synth

UNIT = {"bfloat16": 2.0 ** -9, "float16": 2.0 ** -11}

# H, Hkv, D, page size, pages per sequence, lengths
CASES = [
    (16, 8, 128, 16, 512, [8192, 1, 0, 31, 4097, 33, 8191, 0, 2000]),
    (16, 8, 64, 32, 128, [4096, 17, 0, 0, 1000] + [64] * 27 + [4095]),
    (32, 16, 32, 8, 3300, [0, 2400, 5, 1999, 0]),
    (16, 8, 128, 16, 512, [8192, 7000, 8191, 8192, 7900, 8160, 8001, 8192]),
    (8, 4, 128, 16, 128, [0] * 3 + list(range(1, 140)) + [2048]),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_balanced_paged_decode_matches_the_oracle(torch_gpu, dtype, case):
    torch = torch_gpu
    H, Hkv, D, page, pages, lens = CASES[case]
    B = len(lens)
    q = synth.round_to(synth.uniform(1, (B, H, 1, D)), dtype)
    total = sum(-(-n // page) for n in lens) + 1
    kc, vc = (synth.round_to(synth.uniform(s, (total, page, Hkv, D)), dtype) for s in (2, 3))
    order = np.random.RandomState(case).permutation(total)
    table = np.zeros((B, pages), np.int32)  # past a sequence's end: page 0, never read
    used = 0
    for b, n in enumerate(lens):
        m = -(-n // page)
        table[b, :m] = order[used:used + m]
        used += m
    print(f"[paged balance] {dtype} case {case}", flush=True)
    o, lse = cuflash_attn.flash_attention_decode_paged(
        *(synth.to_torch(x, dtype) for x in (q, kc, vc)), torch.from_numpy(table).cuda(),
        torch.tensor(lens, dtype=torch.int32, device="cuda"), scale=2.0 * D ** -0.5)
    torch.cuda.synchronize()
    o, lse = synth.to_numpy(o), synth.to_numpy(lse)
    for b, n in enumerate(lens):
        if n == 0:
            assert not o[b].any() and np.all(np.isneginf(lse[b]))
            continue
        k, v = (x[table[b, :-(-n // page)]].reshape(-1, Hkv, D)[:n].transpose(1, 0, 2)
                for x in (kc, vc))
        k, v = (np.ascontiguousarray(np.repeat(x, H // Hkv, axis=0))[None] for x in (k, v))
        o_ref, l_ref = oracle.forward(q[b:b + 1], k, v, 2.0 * D ** -0.5, False)
        assert max_abs(o[b:b + 1], o_ref) <= 2.25 * UNIT[dtype], f"O of sequence {b}"
        assert max_abs(lse[b:b + 1], l_ref) <= 2e-5, f"L of sequence {b}"
