"""The attention calls that the speed of this library is measured on.

A case is one call, or one forward and backward pair, of the tensor-level entry points in
cuflash_attn, with new outputs allocated by the call as a program that uses them does. Fields:

  op      "forward"       flash_attention_forward
          "train"         flash_attention_forward, then flash_attention_backward
          "forward_ext"   flash_attention_forward_ext (grouped heads, separate lengths)
          "train_ext"     flash_attention_forward_ext, then flash_attention_backward_ext
          "decode"        flash_attention_decode, one query per head, split count left to the call
          "paged"         flash_attention_decode_paged, the same over a paged cache
  dtype   "float16", "bfloat16" or "float32"
  B, H, Hkv, Nq, Nk, D    batch, query heads, key/value heads, query and key lengths, head_dim
  causal  query i sees the keys j <= i + Nk - Nq
  page    keys per page ("paged" only; Nk is then the longest sequence, and the sequences of a
          batch have the lengths Nk, Nk (B-1)/B, ..., Nk/B in an order of the seed)
  std     standard deviation of the inputs (16-bit types; float32 inputs are uniform in [-1, 1])
"""

import math
import os
import random
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "cuflash-attn_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import cuflash_attn  # noqa: E402


def _case(op, dtype, B, H, Hkv, Nq, Nk, D, causal, page=0, std=1.0, **name):
    return dict(name, op=op, dtype=dtype, B=B, H=H, Hkv=Hkv, Nq=Nq, Nk=Nk, D=D, causal=causal,
                page=page, std=std)


def listed():
    return [
        # The smallest prefill: one short prompt of a small model, where latency counts.
        _case("forward", "float16", 1, 8, 8, 129, 129, 64, True, name="forward_prompt_129"),
        # An encoder's attention without a mask, a batch of ordinary length.
        _case("forward", "float16", 4, 16, 16, 2048, 2048, 64, False,
              name="forward_encoder_2048"),
        # A training step of one short sequence: a small launch in both directions.
        _case("train", "float16", 1, 8, 8, 1024, 1024, 64, True, name="train_short_1024"),
        # Training in single precision.
        _case("train", "float32", 2, 8, 8, 1024, 1024, 64, True, name="train_f32_1024"),
        # The ordinary training step of a language model.
        _case("train", "bfloat16", 2, 16, 16, 4096, 4096, 128, True, name="train_4096"),
        # Training at a long context, the largest product of heads and lengths.
        _case("train", "bfloat16", 1, 32, 32, 16384, 16384, 128, True, std=0.5,
              name="train_long_16384"),
        # Training with grouped heads on a ragged length.
        _case("train_ext", "bfloat16", 2, 16, 4, 2001, 2001, 128, True,
              name="train_grouped_2001"),
        # Training with the widest heads, one row more than whole tiles.
        _case("train_ext", "bfloat16", 1, 16, 16, 2049, 2049, 256, True, name="train_wide_2049"),
        # A few new tokens against a cache: the next turn of a chat, or drafted tokens checked.
        _case("forward_ext", "bfloat16", 1, 32, 8, 61, 8253, 128, True, name="extend_61_of_8253"),
        # The smallest decode: one user, a short context, grouped heads.
        _case("decode", "bfloat16", 1, 32, 8, 1, 1000, 128, False, name="decode_one_1000"),
        # Decode of a batch at a long context, the most bytes.
        _case("decode", "float16", 16, 32, 32, 1, 32768, 128, False, name="decode_batch_32768"),
        # Serving: a batch of sequences of unlike lengths in a paged cache.
        _case("paged", "float16", 16, 32, 8, 1, 8191, 128, False, page=16,
              name="decode_paged_8191"),
    ]


_GROUPED = [(32, 8), (16, 4), (16, 16), (32, 32), (8, 1), (32, 4), (12, 2), (8, 8), (24, 8)]


def _whole(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    while True:
        op = rng.choice(["forward", "train", "forward_ext", "train_ext", "decode", "paged"])
        dtype = rng.choice(["float16", "bfloat16", "bfloat16", "float16", "float32"])
        B = _whole(rng, 1, 16)
        if op in ("forward", "train"):
            H = rng.choice([4, 8, 12, 16, 32])
            N = _whole(rng, 64, 16384)
            c = _case(op, dtype, B, H, H, N, N, rng.choice([32, 64, 128, 128]),
                      rng.random() < 0.7)
        elif op in ("forward_ext", "train_ext"):
            H, Hkv = rng.choice(_GROUPED)
            Nk = _whole(rng, 64, 16384)
            Nq = Nk if rng.random() < 0.5 else _whole(rng, 1 if op == "forward_ext" else 64, Nk)
            c = _case(op, dtype, B, H, Hkv, Nq, Nk, rng.choice([64, 96, 128, 128, 256]),
                      rng.random() < 0.8)
        else:
            H, Hkv = rng.choice(_GROUPED)
            c = _case(op, dtype, B, H, Hkv, 1, _whole(rng, 128, 32768),
                      rng.choice([64, 128, 128]), False,
                      page=rng.choice([16, 32, 64]) if op == "paged" else 0)
        w = work(c)
        # Single precision runs at a sixteenth of the 16-bit matrix rate.
        if w["bytes"] < 8e9 and w["flops"] < (1.5e11 if dtype == "float32" else 3e12):
            return c


def _lengths(c):
    return [max(1, c["Nk"] * (i + 1) // c["B"]) for i in range(c["B"])]


def prepare(c, seed):
    dev = torch.device("cuda")
    dtype = getattr(torch, c["dtype"])
    gen = torch.Generator(device=dev).manual_seed(seed)

    def values(*shape):
        if dtype == torch.float32:
            return torch.rand(shape, device=dev, generator=gen) * 2 - 1
        x = torch.empty(shape, device=dev, dtype=dtype)
        for row in x:  # one batch row (or page) block at a time: float32 copies stay small
            row.copy_(torch.randn(row.shape, device=dev, generator=gen) * c["std"])
        return x

    B, H, Hkv, Nq, Nk, D = (c[k] for k in ("B", "H", "Hkv", "Nq", "Nk", "D"))
    s = {"case": c, "q": values(B, H, Nq, D)}
    if c["op"] == "paged":
        lengths = _lengths(c)
        random.Random(seed).shuffle(lengths)
        pages = -(-Nk // c["page"])
        order = torch.randperm(B * pages, device=dev, generator=gen)
        s["k"], s["v"] = (values(B, pages * c["page"], Hkv, D).view(B * pages, c["page"], Hkv, D)
                          for _ in range(2))
        s["table"] = order.to(torch.int32).view(B, pages)
        s["lengths"] = torch.tensor(lengths, dtype=torch.int32, device=dev)
    else:
        s["k"], s["v"] = (values(B, Hkv, Nk, D) for _ in range(2))
    if c["op"].startswith("train"):
        s["do"] = values(B, H, Nq, D)
    return s


def run(s):
    c = s["case"]
    q, k, v = s["q"], s["k"], s["v"]
    if c["op"] == "decode":
        return cuflash_attn.flash_attention_decode(q, k, v)
    if c["op"] == "paged":
        return cuflash_attn.flash_attention_decode_paged(q, k, v, s["table"], s["lengths"])
    ext = c["op"].endswith("_ext")
    forward, backward = ((cuflash_attn.flash_attention_forward_ext,
                          cuflash_attn.flash_attention_backward_ext) if ext else
                         (cuflash_attn.flash_attention_forward,
                          cuflash_attn.flash_attention_backward))
    o, lse = forward(q, k, v, causal=c["causal"])
    if not c["op"].startswith("train"):
        return o, lse
    return (o, lse) + tuple(backward(q, k, v, o, lse, s["do"], causal=c["causal"]))


def work(c):
    B, H, Hkv, Nq, Nk, D = (c[k] for k in ("B", "H", "Hkv", "Nq", "Nk", "D"))
    size = 4 if c["dtype"] == "float32" else 2
    # Query and key pairs that the mask keeps; 4 D operations each forward, 10 D backward.
    pairs = Nq * Nk - (Nq * (Nq - 1) // 2 if c["causal"] else 0)
    queries, keys = B * H * Nq * D * size, B * Hkv * Nk * D * size
    if c["op"] == "paged":
        pairs = sum(_lengths(c)) / B
        keys = sum(_lengths(c)) * Hkv * D * size
    nbytes = 2 * queries + 2 * keys + B * H * Nq * 4
    flops = 4 * B * H * pairs * D
    if c["op"].startswith("train"):
        # The forward's Q, K, V, O and L count once; dO is read, dQ, dK and dV are written.
        nbytes += 2 * queries + 2 * keys
        flops *= 3.5
    return {"bytes": nbytes, "flops": flops}


def tolerance(c):
    # About four times the distance of the results from exact(): 2.5e-3 for bfloat16 and 3.1e-4
    # for float16, the rounding of the output and of P and dS; up to 8e-7 for float32 at 1024
    # keys, its sums and exponentials, and more where they are longer.
    return {"rel": {"float32": 1e-5, "float16": 1.3e-3, "bfloat16": 1e-2}[c["dtype"]]}


def exact(c, seed):
    s = prepare(c, seed)
    B, H, Hkv, Nq, Nk, D = (c[k] for k in ("B", "H", "Hkv", "Nq", "Nk", "D"))
    train = c["op"].startswith("train")
    scale = D ** -0.5
    q, group = s["q"], H // Hkv
    new = lambda *shape: torch.zeros(shape, device=q.device, dtype=torch.float64)  # noqa: E731
    o, lse = new(B, H, Nq, D), new(B, H, Nq)
    if train:
        dq, dk, dv = new(B, H, Nq, D), new(B, Hkv, Nk, D), new(B, Hkv, Nk, D)
    hidden = None
    if c["causal"]:
        rows = torch.arange(Nq, device=q.device).unsqueeze(1)
        hidden = torch.arange(Nk, device=q.device).unsqueeze(0) > rows + (Nk - Nq)
    for b in range(B):
        if c["op"] == "paged":
            n = int(s["lengths"][b])
            at = s["table"][b].long()
            keys, values = (s[x][at].reshape(-1, Hkv, D)[:n] for x in ("k", "v"))
        for h in range(H):
            if c["op"] == "paged":
                k, v = (x[:, h // group].double() for x in (keys, values))
            else:
                k, v = (s[x][b, h // group].double() for x in ("k", "v"))
            x = q[b, h].double()
            p = torch.mm(x, k.t())
            p *= scale
            if hidden is not None:
                p.masked_fill_(hidden, -math.inf)
            l = torch.logsumexp(p, dim=1)
            p -= l.unsqueeze(1)
            p.exp_()
            o[b, h], lse[b, h] = torch.mm(p, v), l
            if not train:
                continue
            g = s["do"][b, h].double()
            dv[b, h // group] += torch.mm(p.t(), g)
            ds = torch.mm(g, v.t())
            ds -= (g * o[b, h]).sum(1, keepdim=True)
            ds *= p
            ds *= scale
            dq[b, h] = torch.mm(ds, k)
            dk[b, h // group] += torch.mm(ds.t(), x)
    return (o, lse, dq, dk, dv) if train else (o, lse)
