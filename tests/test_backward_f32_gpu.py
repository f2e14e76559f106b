"""The fp32 backward at the sizes where its kernels can go wrong and on both sides of the rule that
chooses them: bwd32_kernel (32-row items whose blocks are spread over four waves) and the kernels
of 128-row items, in one launch and in two.

Expected values: float64 attention and its gradients in plain torch on the same inputs. Bound: the
relative 2-norm error of a sum of n fp32 terms stays below about sqrt(n) * 2^-24 (2.7e-6 at 2048),
doubled for the products and exponentials that enter it.
"""

from __future__ import annotations

import pytest

import cuflash_attn

# B, H, Hkv, Nq, Nk, D, causal
SHAPES = [
    # bwd32_kernel: one block, ragged tiles, fewer blocks than waves, key tiles that no early
    # query sees, grouped heads, every head_dim.
    (1, 1, 1, 1, 1, 64, True),
    (1, 3, 3, 33, 33, 64, True),
    (1, 4, 2, 65, 190, 32, True),
    (2, 6, 2, 97, 160, 96, False),
    (1, 5, 1, 129, 129, 128, True),
    (1, 8, 8, 1001, 1001, 64, True),
    (1, 2, 2, 300, 77, 64, False),
    # 128-row items: both kinds in one launch, then in two.
    (1, 32, 32, 500, 500, 128, False),
    (1, 32, 32, 2017, 2017, 64, False),
]


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "-".join(map(str, s)))
def test_f32_backward_matches_float64(torch_gpu, shape):
    torch = torch_gpu
    B, H, Hkv, Nq, Nk, D, causal = shape
    group, scale = H // Hkv, D ** -0.5
    gen = torch.Generator(device="cuda").manual_seed(sum(shape))
    q, do = (torch.rand((B, H, Nq, D), device="cuda", generator=gen) * 2 - 1 for _ in range(2))
    k, v = (torch.rand((B, Hkv, Nk, D), device="cuda", generator=gen) * 2 - 1 for _ in range(2))
    print(f"[f32 backward] {shape}", flush=True)
    o, lse = cuflash_attn.flash_attention_forward_ext(q, k, v, causal=causal)
    got = cuflash_attn.flash_attention_backward_ext(q, k, v, o, lse, do, causal=causal)
    torch.cuda.synchronize()

    def close(x, ref, what):
        err = float((x.double() - ref).norm() / max(float(ref.norm()), 1e-30))
        # One key: P = 1 and dS = P (dP - D) cancels, exactly 0 but for fp32 rounding.
        if Nk == 1 and what != "dV":
            assert float(x.abs().max()) <= 1e-5, what
        else:
            assert err <= 5.4e-6, f"{what}: {err}"

    mask = None
    if causal:
        mask = torch.arange(Nk, device="cuda") > torch.arange(Nq, device="cuda")[:, None] + Nk - Nq
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
