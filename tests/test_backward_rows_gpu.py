"""The 16-bit backward of small launches (bwd16_rows_kernel).

Such a launch runs one workgroup per 32-row tile whose waves take every eighth (head_dim 96 and
128: fourth) block of the other side. Checked against float64 gradients in plain torch at the
edges: one row and key, ragged tiles, fewer blocks than waves, key tiles that no early query sees,
grouped heads (one key tile over all query heads of its group), every head_dim it takes.

Bound: a gradient is a sum of products with one factor (P or dS) rounded to the input type, and is
rounded once more at the end. A rounding error is spread evenly over at most the unit roundoff u, so
its root mean square is u / sqrt(3); two independent ones give 0.82 u in the relative 2-norm, and
the rounded O that enters D a part of that again. 2 u leaves a factor of two.
"""

from __future__ import annotations

import pytest

import cuflash_attn

UNIT = {"bfloat16": 2.0 ** -9, "float16": 2.0 ** -11}

# B, H, Hkv, Nq, Nk, D, causal
SHAPES = [
    (1, 2, 2, 33, 33, 64, True),
    (1, 4, 2, 65, 190, 32, True),
    (2, 6, 2, 97, 160, 96, False),
    (1, 5, 1, 129, 129, 128, True),
    (1, 8, 8, 1001, 1001, 64, True),
    (1, 4, 4, 700, 700, 128, True),
    (1, 2, 2, 300, 77, 64, False),
    # Several items per CU: grouped heads with few query rows.
    (8, 32, 8, 46, 700, 32, True),
    (7, 24, 8, 40, 900, 128, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_small_backward_matches_float64(torch_gpu, dtype, shape):
    torch = torch_gpu
    B, H, Hkv, Nq, Nk, D, causal = shape
    group, scale = H // Hkv, D ** -0.5
    gen = torch.Generator(device="cuda").manual_seed(sum(shape))
    dt = getattr(torch, dtype)
    q, do = ((torch.rand((B, H, Nq, D), device="cuda", generator=gen) * 2 - 1).to(dt)
             for _ in range(2))
    k, v = ((torch.rand((B, Hkv, Nk, D), device="cuda", generator=gen) * 2 - 1).to(dt)
            for _ in range(2))
    print(f"[small backward] {dtype} {shape}", flush=True)
    o, lse = cuflash_attn.flash_attention_forward_ext(q, k, v, causal=causal)
    got = cuflash_attn.flash_attention_backward_ext(q, k, v, o, lse, do, causal=causal)
    torch.cuda.synchronize()
    mask = None
    if causal:
        mask = torch.arange(Nk, device="cuda") > torch.arange(Nq, device="cuda")[:, None] + Nk - Nq

    def close(x, ref, what):
        err = float((x.double() - ref).norm() / ref.norm())
        assert err <= 2.0 * UNIT[dtype], f"{what}: {err}"

    for hk in sorted({0, Hkv - 1}):
        kd, vd = k[-1, hk].double(), v[-1, hk].double()
        dk, dv = torch.zeros_like(kd), torch.zeros_like(vd)
        for h in range(hk * group, (hk + 1) * group):
            qd, dod = q[-1, h].double(), do[-1, h].double()
            s = qd @ kd.t() * scale
            if mask is not None:
                s = s.masked_fill(mask, float("-inf"))
            p = torch.softmax(s, dim=1)
            dp = dod @ vd.t()
            ds = p * (dp - (p * dp).sum(1, keepdim=True)) * scale
            dv += p.t() @ dod
            dk += ds.t() @ qd
            close(got[0][-1, h], ds @ kd, "dQ")
        close(got[1][-1, hk], dk, "dK")
        close(got[2][-1, hk], dv, "dV")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("head_dim", [32, 64, 96, 128])
def test_nan_reaches_what_sees_it_and_no_other_tile(torch_gpu, dtype, head_dim):
    """A NaN in one row of dO: that row of dQ and every key it sees are NaN; the other rows of dQ,
    and the keys of later 32-key tiles, are as without it, bit for bit."""
    torch = torch_gpu
    dt = getattr(torch, dtype)
    gen = torch.Generator(device="cuda").manual_seed(head_dim)
    q, k, v, do = ((torch.rand((1, 4, 200, head_dim), device="cuda", generator=gen) * 2 - 1).to(dt)
                   for _ in range(4))
    o, lse = cuflash_attn.flash_attention_forward_ext(q, k, v, causal=True)
    clean = cuflash_attn.flash_attention_backward_ext(q, k, v, o, lse, do, causal=True)
    row = 100
    do[:, :, row, 3] = float("nan")
    dq, dk, dv = cuflash_attn.flash_attention_backward_ext(q, k, v, o, lse, do, causal=True)
    torch.cuda.synchronize()
    others = torch.arange(200, device="cuda") != row
    assert torch.equal(dq[:, :, others], clean[0][:, :, others])
    assert bool(dq[:, :, row].isnan().all())
    assert torch.equal(dk[:, :, 128:], clean[1][:, :, 128:])
    assert torch.equal(dv[:, :, 128:], clean[2][:, :, 128:])
    assert bool(dk[:, :, :row + 1].isnan().all()) and bool(dv[:, :, :row + 1, 3].isnan().all())
