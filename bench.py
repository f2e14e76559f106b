#!/usr/bin/env python3
"""Headline benchmark of libcuflash_attn on one MI355X.

Metric: "fwd+bwd TFLOP/s (bf16 causal N=4096 D=128) + decode HBM GB/s at 32k KV".

* A step is one forward + one backward pass of config 3 (bf16, causal, B=2 H=16 N=4096 D=128,
  scale 1/sqrt(128), Q/K/V/dO i.i.d. N(0,1) from seeds 1-4) on inputs resident in HBM.
  value = (F_fwd + F_bwd) / step time with the reference's FLOP model
  (benchmarks/bench_flash_attention.cu:34-44, causal x0.5 at :457-460):
  F_fwd = 4 B H N^2 D / 2, F_bwd = 2.5 F_fwd.
* The K timed steps (default 100) run as five consecutive regions of K/5 steps (events between
  them, one synchronized bracket around all of them); ms_per_step is the median region's time
  per step.
* Decode (config 4: fp16, B=16 H=32, 1 query, 32768 keys, D=128) is timed for 16/32/64 splits
  (the headline: the best of these, config 4's range) and the library's automatic choice
  (reported beside it); GB/s counts K and V read once plus Q read, O and L written.
* roofline: the dominant kernel of the step against MI355X's dense bf16 MFMA peak, timed live on
  the launch stream: the forward from back-to-back forward calls between two HIP events, the
  backward's main kernel from back-to-back backward calls minus the delta kernel's time (HIP
  events around each of its launches, cuflash_profile_enable). `rooflines` lists each kernel
  with the per-launch event-pair figure beside it; `traffic` is the committed rocprofv3
  FETCH_SIZE / WRITE_SIZE figure (profiles/hbm_traffic_pmc.md), not a measurement of this run.
* ext: the extended forward / backward (cuflash_attention_{forward,backward}_ext_bf16) on a
  prefill chunk against a KV cache with grouped-query heads, grouped-query training at the
  config-3 size, and head_dim 96 and 256 at the config-3 size; reported beside the headline.
* sdpa: this library against torch.nn.functional.scaled_dot_product_attention on the same GPU,
  restricted to its fused flash / memory-efficient kernels: the forward at the shapes of the
  reference's own SDPA comparison (fp16 causal head_dim 64, docs/performance/benchmarks.md:
  106-114, where the reference reaches 0.42-0.67x of SDPA on an A100), and config 3's forward +
  backward; reported beside the headline (speedup = SDPA time / this library's time).
* reference_shapes: this library's forward and backward at the shapes of the reference's published
  timing tables (fp16 causal head_dim 64, docs/performance/benchmarks.md:60-96, NVIDIA GPUs,
  v0.4.0 snapshot), with those published times beside them as context.
* decode_graph: a launch-bound serving step (16 decode calls of 1 sequence, 32 heads, 1024 keys,
  head_dim 128, fp16) launched eagerly and replayed from captured HIP graphs of the allocating
  entry point and of the one that allocates nothing: time per call.
* cpu_baseline: the reference's naive O(N^2) CPU attention (tests/unit/test_forward.cu:21-118,
  tests/unit/test_backward.cu:21-127) restated in C, float arithmetic, on this box's host cores
  (the threads used and sched_getaffinity's count are both printed): whole heads of config 3
  itself at N=4096 (scaled by B*H / heads), one thread on every 16th row of one head, and 16 of
  config 4's decode rows; see cpu_baseline().

Before the W warmup steps the step runs untimed for --ramp-ms (default 1 s): the first few dozen
steps after the inputs are written run 5-10% slower while the GPU's clock settles.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--ramp-ms MS] [--no-cpu-baseline]
                      [--no-decode] [--no-ext] [--no-configs] [--no-sdpa]
                      [--no-reference-shapes] [--no-decode-graph]
"""

from __future__ import annotations

import argparse
import json
import os
import sys
import time

REPO = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(REPO, "cuflash-attn_amd"))
sys.path.insert(0, REPO)

PEAK_BF16_TFLOPS = 2516.6  # MI355X dense bf16 MFMA
PEAK_HBM_GBS = 8000.0      # MI355X HBM3E
PEAK_FP32_TFLOPS = 157.3   # MI355X dense fp32 (MFMA)

CFG3 = dict(B=2, H=16, N=4096, D=128, causal=True)
CFG4 = dict(B=16, H=32, LKV=32768, D=128)


def flops_fwd(B, H, N, D, causal):
    return 4.0 * B * H * N * N * D * (0.5 if causal else 1.0)


def decode_bytes(B, H, LKV, D, elem=2):
    return B * H * D * (2 * LKV + 2) * elem + B * H * 4


TRAFFIC_FILE = os.path.join(REPO, "profiles", "hbm_traffic_pmc.md")


def committed_traffic(kernel_label):
    """HBM bytes per launch of `kernel_label` from the committed rocprofv3 PMC summary (lines
    `traffic: <label> <bytes>`), or None when that kernel has no committed measurement."""
    try:
        with open(TRAFFIC_FILE) as f:
            for line in f:
                parts = line.split()
                if len(parts) == 3 and parts[0] == "traffic:" and parts[1] == kernel_label:
                    return int(parts[2])
    except OSError:
        pass
    return None


def pmc_workload(kind):
    """Short fixed workloads for rocprofv3 --pmc passes (no timing, no output line):
    cfg3 = 2 x (forward + backward) of config 3; cfg1 / cfg2 = 2 x the forward of config 1 / 2;
    cfg5 = 1 x (forward + backward) of config 5; decode = 2 x config-4 decode (auto splits);
    decode_gqa / decode_paged = 2 x the grouped-query decode at config-4 size (32 query heads
    over 8 key/value heads; contiguous / 16-key pages in shuffled order); copy = one
    device-to-device copy of 1 GiB, the calibration kernel for FETCH_SIZE and WRITE_SIZE."""
    import torch

    import cuflash_attn

    dev = torch.device("cuda:0")
    if kind == "copy":
        a = torch.ones(1 << 28, device=dev, dtype=torch.float32)
        b = torch.empty_like(a)
        b.copy_(a)
    elif kind == "cfg3":
        c = CFG3
        xs = [torch.randn((c["B"], c["H"], c["N"], c["D"]), device=dev).to(torch.bfloat16)
              for _ in range(4)]
        for _ in range(2):
            o, lse = cuflash_attn.flash_attention_forward(*xs[:3], causal=True)
            cuflash_attn.flash_attention_backward(*xs[:3], o, lse, xs[3], causal=True)
    elif kind in ("cfg1", "cfg2", "cfg5"):
        name, sfx, B, H, N, D, causal, with_bwd, dist = next(
            w for w in CONFIG_WORKLOADS if w[0] == kind)
        dt = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}[sfx]
        std = 0.5 if dist == "N(0,0.5)" else 1.0
        xs = [(torch.randn((B, H, N, D), device=dev) * std).to(dt) for _ in range(4)]
        for _ in range(1 if with_bwd else 2):
            o, lse = cuflash_attn.flash_attention_forward(*xs[:3], causal=causal)
            if with_bwd:
                cuflash_attn.flash_attention_backward(*xs[:3], o, lse, xs[3], causal=causal)
    elif kind == "decode":
        c = CFG4
        q = torch.randn((c["B"], c["H"], 1, c["D"]), device=dev).half()
        k = torch.randn((c["B"], c["H"], c["LKV"], c["D"]), device=dev, dtype=torch.float16)
        v = torch.randn_like(k)
        for _ in range(2):
            cuflash_attn.flash_attention_decode(q, k, v, num_splits=0)
    elif kind in ("decode_gqa", "decode_paged"):
        c = CFG4
        hkv, page = 8, 16
        q = torch.randn((c["B"], c["H"], 1, c["D"]), device=dev).half()
        k = torch.randn((c["B"], hkv, c["LKV"], c["D"]), device=dev, dtype=torch.float16)
        v = torch.randn_like(k)
        if kind == "decode_gqa":
            for _ in range(2):
                cuflash_attn.flash_attention_decode(q, k, v, num_splits=0)
        else:
            npages = c["B"] * c["LKV"] // page
            g = torch.Generator(device=dev)
            g.manual_seed(6)
            perm = torch.randperm(npages, generator=g, device=dev)
            kp, vp = (t.reshape(c["B"], hkv, c["LKV"] // page, page, c["D"]).permute(0, 2, 3, 1, 4)
                      .reshape(npages, page, hkv, c["D"])[perm].contiguous() for t in (k, v))
            del k, v
            table = torch.argsort(perm).to(torch.int32).reshape(c["B"], -1).contiguous()
            lens = torch.full((c["B"],), c["LKV"], dtype=torch.int32, device=dev)
            for _ in range(2):
                cuflash_attn.flash_attention_decode_paged(q, kp, vp, table, lens, num_splits=0)
    torch.cuda.synchronize()
    return 0


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--ramp-ms", type=float, default=1000.0,
                    help="untimed steps for at least this long before the warmup steps, so that "
                         "the GPU reaches its steady clock (default 1000 ms)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-decode", action="store_true")
    ap.add_argument("--no-parity", action="store_true")
    ap.add_argument("--no-ext", action="store_true")
    ap.add_argument("--no-sdpa", action="store_true")
    ap.add_argument("--no-reference-shapes", action="store_true")
    ap.add_argument("--no-decode-graph", action="store_true")
    ap.add_argument("--no-configs", action="store_true")
    ap.add_argument("--pmc-workload", choices=("cfg1", "cfg2", "cfg3", "cfg5", "decode", "decode_gqa",
                                               "decode_paged", "copy"),
                    default=None,
                    help="run only a short fixed workload for rocprofv3 --pmc passes")
    ap.add_argument("--cpu-seconds", type=float, default=8.0,
                    help="wall time the multi-threaded CPU-baseline sample aims for: whole "
                         "config-3 heads are timed one after another until this much time has "
                         "passed (at most 8 heads; default 8 s)")
    return ap.parse_args()


def causal_pairs(nq, nk):
    """(query, key) pairs a bottom-right aligned causal mask keeps: query i sees i + nk - nq + 1
    keys."""
    return nq * (nk - nq) + nq * (nq + 1) / 2


EXT_WORKLOADS = [
    # name, B, H, Hkv, q_len, kv_len, D, backward too
    ("prefill_chunk_gqa", 1, 32, 8, 2048, 16384, 128, False),
    ("gqa_train", 2, 16, 4, 4096, 4096, 128, True),
    ("head_dim_96", 2, 16, 16, 4096, 4096, 96, True),
    ("head_dim_256", 2, 16, 16, 4096, 4096, 256, True),
]


# The reference's SDPA comparison shapes (docs/performance/benchmarks.md:106-114): fp16, causal,
# head_dim 64, (batch, heads, seq_len).
SDPA_SHAPES = [(1, 8, 1024), (8, 16, 1024), (1, 8, 4096), (8, 16, 4096), (1, 8, 8192),
               (8, 16, 8192), (1, 8, 16384)]


def bench_sdpa(torch, steps):
    """Forward (and config 3's forward + backward, config 4's decode) against torch's
    scaled_dot_product_attention with only its fused flash / memory-efficient kernels allowed
    (never the math path), as the median of five regions of `steps` calls each, events on the
    current stream."""
    import torch.nn.functional as F
    from torch.nn.attention import SDPBackend, sdpa_kernel

    import cuflash_attn

    dev = torch.device("cuda:0")
    fused = [SDPBackend.FLASH_ATTENTION, SDPBackend.EFFICIENT_ATTENTION]

    def median_ms(fn):
        for _ in range(3):
            fn()
        torch.cuda.synchronize()
        times = []
        for _ in range(5):
            e0 = torch.cuda.Event(enable_timing=True)
            e1 = torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(steps):
                fn()
            e1.record()
            torch.cuda.synchronize()
            times.append(e0.elapsed_time(e1) / steps)
        return sorted(times)[2]

    out = {"torch": torch.__version__, "backends": "flash / memory-efficient only",
           "reference_on_a100": "0.42x-0.67x of SDPA (forward, these shapes)", "forward": []}
    try:
        with sdpa_kernel(fused):
            for B, H, N in SDPA_SHAPES:
                q, k, v = (torch.randn((B, H, N, 64), device=dev, dtype=torch.float16)
                           for _ in range(3))
                ours = median_ms(lambda: cuflash_attn.flash_attention_forward(q, k, v,
                                                                              causal=True))
                ref = median_ms(lambda: F.scaled_dot_product_attention(q, k, v, is_causal=True))
                out["forward"].append({"batch": B, "heads": H, "seq_len": N,
                                       "ours_ms": round(ours, 4), "sdpa_ms": round(ref, 4),
                                       "speedup": round(ref / ours, 2)})
            c = CFG3
            q, k, v, do = (torch.randn((c["B"], c["H"], c["N"], c["D"]), device=dev,
                                       dtype=torch.bfloat16) for _ in range(4))

            def ours_step():
                o, lse = cuflash_attn.flash_attention_forward(q, k, v, causal=True)
                cuflash_attn.flash_attention_backward(q, k, v, o, lse, do, causal=True)

            qg, kg, vg = (t.detach().clone().requires_grad_(True) for t in (q, k, v))

            def sdpa_step():
                o = F.scaled_dot_product_attention(qg, kg, vg, is_causal=True)
                torch.autograd.grad(o, (qg, kg, vg), do)

            ours = median_ms(ours_step)
            ref = median_ms(sdpa_step)
            out["cfg3_fwd_bwd"] = {"workload": "bf16 causal B=2 H=16 N=4096 D=128",
                                   "ours_ms": round(ours, 4), "sdpa_ms": round(ref, 4),
                                   "speedup": round(ref / ours, 2)}
            del q, k, v, do, qg, kg, vg
            c = CFG4
            q = torch.randn((c["B"], c["H"], 1, c["D"]), device=dev, dtype=torch.float16)
            k, v = (torch.randn((c["B"], c["H"], c["LKV"], c["D"]), device=dev,
                                dtype=torch.float16) for _ in range(2))
            ours = median_ms(lambda: cuflash_attn.flash_attention_decode(q, k, v, num_splits=16))
            ref = median_ms(lambda: F.scaled_dot_product_attention(q, k, v))
            out["cfg4_decode"] = {"workload": "fp16 B=16 H=32 Lkv=32768 D=128, one query "
                                              "(this library at 16 splits)",
                                  "ours_ms": round(ours, 4), "sdpa_ms": round(ref, 4),
                                  "speedup": round(ref / ours, 2)}
            del q, k, v
    except RuntimeError as e:  # no fused SDPA kernel for these inputs on this build of torch
        out["unavailable"] = str(e)[:200]
    return out


# The reference's published timing tables (docs/performance/benchmarks.md:60-96; fp16, causal,
# head_dim 64): (batch, heads, seq_len) -> forward ms on A100 / H100, backward ms on A100.
REFERENCE_SHAPES = [
    ((1, 8, 1024), {"A100": 0.19, "H100": 0.11}, {"A100": 0.41}),
    ((1, 8, 4096), {"A100": 2.18, "H100": 1.15}, {"A100": 4.75}),
    ((1, 8, 8192), {"A100": 7.80, "H100": 3.85}, {"A100": 17.20}),
    ((1, 8, 16384), {"A100": 28.5, "H100": 13.2}, {"A100": 63.5}),
    ((16, 16, 4096), {"A100": 65.60, "H100": 34.50}, None),
    ((1, 16, 32768), {"A100": 205.0, "H100": 88.0}, None),
]


def bench_reference_shapes(torch, steps):
    """Forward (and backward where the reference publishes one) at the reference's published
    shapes, median of five regions of `steps` calls, events on the current stream."""
    import cuflash_attn

    dev = torch.device("cuda:0")

    def median_ms(fn):
        fn()
        torch.cuda.synchronize()
        times = []
        for _ in range(5):
            e0 = torch.cuda.Event(enable_timing=True)
            e1 = torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(steps):
                fn()
            e1.record()
            torch.cuda.synchronize()
            times.append(e0.elapsed_time(e1) / steps)
        return sorted(times)[2]

    rows = []
    for (B, H, N), ref_fwd, ref_bwd in REFERENCE_SHAPES:
        q, k, v, do = (torch.randn((B, H, N, 64), device=dev, dtype=torch.float16)
                       for _ in range(4))
        o, lse = cuflash_attn.flash_attention_forward(q, k, v, causal=True)
        row = {"batch": B, "heads": H, "seq_len": N,
               "fwd_ms": round(median_ms(
                   lambda: cuflash_attn.flash_attention_forward(q, k, v, causal=True)), 4),
               "reference_fwd_ms": ref_fwd}
        if ref_bwd:
            row["bwd_ms"] = round(median_ms(lambda: cuflash_attn.flash_attention_backward(
                q, k, v, o, lse, do, causal=True)), 4)
            row["reference_bwd_ms"] = ref_bwd
        rows.append(row)
        del q, k, v, do, o, lse
    return {"note": "the reference's published times are for fp16 causal head_dim 64 on NVIDIA "
                    "GPUs (v0.4.0 snapshot, docs/performance/benchmarks.md:60-96), reported "
                    "as context", "rows": rows}


def bench_decode_graph(lib, torch, steps):
    """Per-call time of a launch-bound serving step, 16 small decode calls (distinct inputs per
    call, as the layers of a step would have), launched eagerly, replayed from a captured graph of
    the allocating entry point (each captured call records its workspace as a graph allocation and
    free) and replayed from a captured graph of the entry point that allocates nothing; median of
    five regions of `steps` steps each."""
    import ctypes

    import cuflash_attn

    dev = torch.device("cuda:0")
    calls, B, H, L, D = 16, 1, 32, 1024, 128
    qs = [torch.randn((B, H, 1, D), device=dev, dtype=torch.float16) for _ in range(calls)]
    ks = [torch.randn((B, H, L, D), device=dev, dtype=torch.float16) for _ in range(calls)]
    vs = [torch.randn((B, H, L, D), device=dev, dtype=torch.float16) for _ in range(calls)]
    outs = [(torch.empty_like(q), torch.empty((B, H, 1), device=dev, dtype=torch.float32))
            for q in qs]
    noalloc = lib.library.cuflash_attention_decode_noalloc_f16
    noalloc.argtypes = [ctypes.c_void_p] * 5 + [ctypes.c_int] * 4 + [ctypes.c_float,
                                                                     ctypes.c_int, ctypes.c_void_p]
    noalloc.restype = ctypes.c_int

    def step_alloc():
        for q, k, v, (o, lse) in zip(qs, ks, vs, outs):
            cuflash_attn.flash_attention_decode(q, k, v, out=o, lse=lse)

    def step_noalloc():
        sp = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        for q, k, v, (o, lse) in zip(qs, ks, vs, outs):
            st = noalloc(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(),
                         B, H, L, D, D ** -0.5, 0, sp)
            if st != 0:
                raise RuntimeError(f"decode_noalloc status {st}")

    def median_ms(fn):
        fn()
        torch.cuda.synchronize()
        times = []
        for _ in range(5):
            e0 = torch.cuda.Event(enable_timing=True)
            e1 = torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(steps):
                fn()
            e1.record()
            torch.cuda.synchronize()
            times.append(e0.elapsed_time(e1) / steps)
        return sorted(times)[2]

    def captured(fn):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            fn()
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            fn()
        return graph

    res = {"workload": f"{calls} decode calls: fp16 B={B} H={H} Lkv={L} D={D}, auto splits",
           "eager_us_per_call": round(median_ms(step_alloc) * 1e3 / calls, 2)}
    step_alloc()
    torch.cuda.synchronize()
    ref = [(o.clone(), lse.clone()) for o, lse in outs]
    for name, fn in (("graph_allocating", step_alloc), ("graph_noalloc", step_noalloc)):
        graph = captured(fn)
        res[name + "_us_per_call"] = round(median_ms(graph.replay) * 1e3 / calls, 2)
        for o, lse in outs:
            o.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        res[name + "_equals_eager"] = all(torch.equal(o, r[0]) and torch.equal(lse, r[1])
                                          for (o, lse), r in zip(outs, ref))
        del graph
    return res


def bench_ext(lib, torch, steps, stream):
    """Times the extended entry points (bf16, causal) on EXT_WORKLOADS: per-launch forward and
    backward time from the event hook, TFLOP/s with the reference's FLOP model over the (query,
    key) pairs the mask keeps (forward 4 D per pair, backward 2.5 times that)."""
    dev = torch.device("cuda:0")
    fwd = lib.fn("forward_ext", "bf16")
    bwd = lib.fn("backward_ext", "bf16")
    sp = stream.cuda_stream
    out = {}
    for name, B, H, Hkv, nq, nk, D, with_bwd in EXT_WORKLOADS:
        q = torch.randn((B, H, nq, D), device=dev).to(torch.bfloat16)
        k = torch.randn((B, Hkv, nk, D), device=dev).to(torch.bfloat16)
        v = torch.randn((B, Hkv, nk, D), device=dev).to(torch.bfloat16)
        do = torch.randn((B, H, nq, D), device=dev).to(torch.bfloat16)
        o, lse = torch.empty_like(q), torch.empty((B, H, nq), device=dev, dtype=torch.float32)
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        scale = D ** -0.5

        def run():
            st = fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), B, H,
                     Hkv, nq, nk, D, scale, True, sp)
            if with_bwd:
                st |= bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                          lse.data_ptr(), do.data_ptr(), dq.data_ptr(), dk.data_ptr(),
                          dv.data_ptr(), B, H, Hkv, nq, nk, D, scale, True, sp)
            if st != 0:
                raise RuntimeError(f"{name}: library status {st}")

        for _ in range(2):
            run()
        torch.cuda.synchronize()
        lib.profile_enable(True)
        for _ in range(steps):
            run()
        torch.cuda.synchronize()
        rep = lib.profile_report()
        lib.profile_enable(False)
        f_fwd = 4.0 * B * H * D * causal_pairs(nq, nk)
        suffix = f"_bf16_d{D}"
        k_ms = {lab[:-len(suffix)]: tot / n for lab, (n, tot) in rep.items()
                if lab.endswith(suffix) and n}
        rec = {"workload": f"bf16 causal B={B} H={H} Hkv={Hkv} q_len={nq} kv_len={nk} D={D}",
               "fwd_ms": round(k_ms["forward"], 4),
               "fwd_tflops": round(f_fwd / (k_ms["forward"] * 1e-3) / 1e12, 1)}
        rec["fwd_frac"] = round(rec["fwd_tflops"] / PEAK_BF16_TFLOPS, 4)
        if with_bwd:
            b_ms = sum(v2 for k2, v2 in k_ms.items() if k2.startswith("backward"))
            rec["bwd_ms"] = round(b_ms, 4)
            rec["bwd_tflops"] = round(2.5 * f_fwd / (b_ms * 1e-3) / 1e12, 1)
            rec["bwd_frac"] = round(rec["bwd_tflops"] / PEAK_BF16_TFLOPS, 4)
            rec["step_tflops"] = round(3.5 * f_fwd / ((k_ms["forward"] + b_ms) * 1e-3) / 1e12, 1)
        out[name] = rec
        log(f"ext {name}: {rec}")
        del q, k, v, do, o, lse, dq, dk, dv
        torch.cuda.empty_cache()
    return out


CONFIG_WORKLOADS = [
    # name, dtype suffix, B, H, N, D, causal, backward too, input distribution
    ("cfg1", "f32", 2, 8, 1024, 64, True, False, "uniform[-1,1]"),
    ("cfg2", "f16", 4, 16, 2048, 64, False, False, "N(0,1)"),
    ("cfg5", "bf16", 1, 32, 16384, 128, True, True, "N(0,0.5)"),
]


def bench_configs(lib, torch, steps, stream):
    """Times BASELINE configurations 1, 2 and 5 through the reference entry points
    (cuflash_attention_{forward,backward}_{f32,f16,bf16}): per-launch times from the event hook,
    TFLOP/s with the reference's FLOP model, fraction of the dense peak of the compute type
    (fp32 MFMA for config 1). Inputs are synthetic, from torch's GPU generator."""
    dev = torch.device("cuda:0")
    dtypes = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
    sp = stream.cuda_stream
    out = {}
    for name, sfx, B, H, N, D, causal, with_bwd, dist in CONFIG_WORKLOADS:
        dt = dtypes[sfx]
        gen = torch.Generator(device=dev)
        gen.manual_seed(1)

        def draw():
            if dist.startswith("uniform"):
                x = torch.rand((B, H, N, D), device=dev, generator=gen) * 2 - 1
            else:
                x = torch.randn((B, H, N, D), device=dev, generator=gen)
                if dist == "N(0,0.5)":
                    x = x * 0.5
            return x.to(dt)

        q, k, v, do = draw(), draw(), draw(), draw()
        o, lse = torch.empty_like(q), torch.empty((B, H, N), device=dev, dtype=torch.float32)
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        scale = D ** -0.5
        fwd = lib.fn("forward", sfx)
        bwd = lib.fn("backward", sfx)

        def run():
            st = fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), B, H,
                     N, D, scale, causal, sp)
            if with_bwd:
                st |= bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                          lse.data_ptr(), do.data_ptr(), dq.data_ptr(), dk.data_ptr(),
                          dv.data_ptr(), B, H, N, D, scale, causal, sp)
            if st != 0:
                raise RuntimeError(f"{name}: library status {st}")

        for _ in range(2):
            run()
        torch.cuda.synchronize()
        lib.profile_enable(True)
        for _ in range(steps):
            run()
        torch.cuda.synchronize()
        rep = lib.profile_report()
        lib.profile_enable(False)
        peak = PEAK_FP32_TFLOPS if sfx == "f32" else PEAK_BF16_TFLOPS
        f_fwd = flops_fwd(B, H, N, D, causal)
        suffix = f"_{sfx}_d{D}"
        k_ms = {lab[:-len(suffix)]: tot / n for lab, (n, tot) in rep.items()
                if lab.endswith(suffix) and n}
        rec = {"workload": f"{sfx} {'causal' if causal else 'non-causal'} B={B} H={H} N={N} "
                           f"D={D}, inputs {dist}",
               "fwd_ms": round(k_ms["forward"], 4),
               "fwd_tflops": round(f_fwd / (k_ms["forward"] * 1e-3) / 1e12, 2),
               "peak_tflops": peak}
        rec["fwd_frac"] = round(rec["fwd_tflops"] / peak, 4)
        if with_bwd:
            b_ms = sum(v2 for k2, v2 in k_ms.items() if k2.startswith("backward"))
            rec["bwd_ms"] = round(b_ms, 4)
            rec["bwd_tflops"] = round(2.5 * f_fwd / (b_ms * 1e-3) / 1e12, 1)
            rec["bwd_frac"] = round(rec["bwd_tflops"] / peak, 4)
            rec["step_tflops"] = round(3.5 * f_fwd / ((k_ms["forward"] + b_ms) * 1e-3) / 1e12, 1)
        out[name] = rec
        log(f"config {name}: {rec}")
        del q, k, v, do, o, lse, dq, dk, dv
        torch.cuda.empty_cache()
    return out


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def host_cpus():
    """Host CPUs this process may run on (sched_getaffinity), uncapped."""
    try:
        return len(os.sched_getaffinity(0))
    except AttributeError:  # pragma: no cover
        return os.cpu_count() or 1


def host_threads():
    """Threads of the CPU-side work: the host CPUs, at most 16."""
    return max(1, min(16, host_cpus()))


def cpu_baseline(host, B, H, N, D, scale, causal, target_s, with_decode):
    """The reference's naive O(N^2) fp32 CPU attention (tests/unit/test_forward.cu:21-118 and
    tests/unit/test_backward.cu:21-127, restated in oracle.c) timed on this box's host cores on
    a bounded sample of the config-3 workload itself, and on a sample of config 4.

    Config 3: whole heads of the timed GPU inputs (the same bf16 values, as float32), each
    head's forward + backward split by query rows over the threads (oracle.naive_rows_f32:
    row i's loops exactly as in the naive code), timed head after head until `target_s` has
    passed (at most 8 heads), then scaled by B * H / heads. One thread: every 16th query row of
    one head, scaled by N / rows (the naive loops do almost the same work for every row: all N
    keys, except the score dot products of masked keys) and by B * H. The rates use the GPU
    line's FLOP model, so gpu_speedup compares the same problem.
    Config 4: 16 of its 512 (batch, head) rows at 32768 keys (fp32 copies of N(0,1) data),
    median of 5 calls; GB/s counts config 4's algorithmic (fp16) bytes of those rows."""
    import numpy as np

    import oracle

    threads = host_threads()
    f_total = 3.5 * flops_fwd(B, H, N, D, causal)
    heads = [(b, h) for b in range(B) for h in range(H)]
    rows_all = np.arange(N, dtype=np.int64)
    log(f"CPU baseline: naive fp32 fwd+bwd, config-3 heads at N={N}, {threads} threads")
    secs, done = 0.0, 0
    for (b, h) in heads[:8]:
        xs = [x[b, h] for x in host]
        c0 = time.perf_counter()
        oracle.naive_rows_f32(xs[0], xs[1], xs[2], xs[3], scale, causal, rows_all,
                              nthreads=threads)
        secs += time.perf_counter() - c0
        done += 1
        if secs >= target_s:
            break
    t_est = secs * (B * H) / done
    cpu = {"value": round(f_total / t_est / 1e12, 6), "unit": "TFLOP/s", "cores": threads,
           "host_cpus": host_cpus(), "kind": "port", "seconds": round(secs, 2),
           "est_seconds_full_workload": round(t_est, 1),
           "sample": f"config 3 itself (bf16 causal B={B} H={H} N={N} D={D}, the timed GPU "
                     f"inputs as float32): {done} of its {B * H} heads, all {N} query rows, "
                     f"forward + backward in the naive fp32 loops of the reference's CPU "
                     f"attention (test_forward.cu:21-118, test_backward.cu:21-127), query rows "
                     f"split over {threads} threads; time scaled by {B * H}/{done}; same FLOP "
                     f"model as the GPU line"}
    rows1 = np.arange(8, N, 16, dtype=np.int64)
    xs = [x[0, 0] for x in host]
    c0 = time.perf_counter()
    oracle.naive_rows_f32(xs[0], xs[1], xs[2], xs[3], scale, causal, rows1, nthreads=1)
    s1 = time.perf_counter() - c0
    t1_est = s1 * (N / rows1.size) * B * H
    cpu["single_thread"] = {
        "value": round(f_total / t1_est / 1e12, 6), "unit": "TFLOP/s", "cores": 1,
        "seconds": round(s1, 2), "est_seconds_full_workload": round(t1_est, 1),
        "sample": f"every 16th query row ({rows1.size} rows) of head (0, 0) of config 3, one "
                  f"thread, the same loops; time scaled by {N}/{rows1.size} and by {B * H} heads"}
    if with_decode:
        Bd, Hd, LKV, Dd = CFG4["B"], CFG4["H"], CFG4["LKV"], CFG4["D"]
        nrow = 16
        log(f"CPU baseline: naive fp32 decode, {nrow} of {Bd * Hd} rows at {LKV} keys")
        rng = np.random.default_rng(4)
        qd = rng.standard_normal((nrow, Dd), dtype=np.float32)
        kd = rng.standard_normal((nrow, LKV, Dd), dtype=np.float32)
        vd = rng.standard_normal((nrow, LKV, Dd), dtype=np.float32)
        times = []
        for _ in range(5):
            c0 = time.perf_counter()
            oracle.naive_decode_f32(qd, kd, vd, Dd ** -0.5, nthreads=threads)
            times.append(time.perf_counter() - c0)
        td = sorted(times)[2]
        nbytes = decode_bytes(Bd, Hd, LKV, Dd) * nrow / (Bd * Hd)
        cpu["decode"] = {
            "value": round(nbytes / td / 1e9, 2), "unit": "GB/s", "cores": threads,
            "seconds": round(td, 4),
            "sample": f"{nrow} of config 4's {Bd * Hd} (batch, head) rows, 1 query against "
                      f"{LKV} keys, D={Dd}, naive fp32 loops (the reference's naive forward at "
                      f"a query length of 1), rows over {threads} threads, median of 5 calls; "
                      f"bytes = config 4's algorithmic fp16 bytes of those rows"}
        del kd, vd
    return cpu


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only; --gpus {args.gpus} is not supported (every "
              "kernel here runs on a single MI355X; sharding over heads or keys across GPUs "
              "is not built)", file=sys.stderr)
        return 2

    if args.pmc_workload:
        return pmc_workload(args.pmc_workload)

    import numpy as np
    import torch

    import cuflash_attn
    from cuflash_attn import synth

    if not torch.cuda.is_available():
        print("no GPU visible", file=sys.stderr)
        return 1
    lib = cuflash_attn.load_library()
    dev = torch.device("cuda:0")
    stream = torch.cuda.current_stream()

    # ---------------- config 3: fwd + bwd ----------------
    B, H, N, D, causal = CFG3["B"], CFG3["H"], CFG3["N"], CFG3["D"], CFG3["causal"]
    scale = D ** -0.5
    shape = (B, H, N, D)
    log("generating config-3 inputs")
    host = [synth.round_to(synth.normal(s, shape), "bfloat16") for s in (1, 2, 3, 4)]
    q, k, v, do = (synth.to_torch(x, "bfloat16", dev) for x in host)
    o = torch.empty_like(q)
    lse = torch.empty((B, H, N), device=dev, dtype=torch.float32)
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    fwd = lib.fn("forward", "bf16")
    bwd = lib.fn("backward", "bf16")
    sp = stream.cuda_stream

    def step():
        st = fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), B, H, N,
                 D, scale, causal, sp)
        st |= bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(),
                  do.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), B, H, N, D, scale,
                  causal, sp)
        if st != 0:
            raise RuntimeError(f"library status {st}")

    # Steady state first: the first few dozen steps after the inputs are generated run 5-10%
    # slower (clock and power ramp), which no fixed small warmup count covers.
    log(f"ramp {args.ramp_ms:.0f} ms, then warmup {args.warmup}")
    ramp_steps = 0
    r0 = time.perf_counter()
    while (time.perf_counter() - r0) * 1e3 < args.ramp_ms:
        for _ in range(10):
            step()
        torch.cuda.synchronize()
        ramp_steps += 10
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()

    # Exactly K timed steps in one bracket (synchronize on both sides), split into up to five
    # consecutive regions by events on the launch stream; the headline is the median region's
    # time per step, so one slow region (clock dip, host hiccup) does not move it.
    nreg = max(1, min(5, args.steps))
    sizes = [args.steps // nreg + (1 if i < args.steps % nreg else 0) for i in range(nreg)]
    log(f"timing {args.steps} steps in {nreg} regions {sizes}")
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(nreg + 1)]
    t0, t1 = ev[0], ev[-1]
    torch.cuda.synchronize()
    ev[0].record(stream)
    for i, n_i in enumerate(sizes):
        for _ in range(n_i):
            step()
        ev[i + 1].record(stream)
    torch.cuda.synchronize()
    region_ms = [ev[i].elapsed_time(ev[i + 1]) / n_i for i, n_i in enumerate(sizes)]
    ms_per_step = float(np.median(region_ms))
    ms_per_step_mean = ev[0].elapsed_time(ev[-1]) / args.steps

    # Per-kernel durations. The forward is one kernel per call: K forward calls back to back
    # between two events give its time per launch directly. A backward call is
    # delta_ld_kernel then bwd_fused_kernel: K backward calls back to back give their sum, and
    # the dominant kernel's time is that minus the delta kernel's, which comes from a pass with
    # the per-launch event hook (events around every launch; they add a few microseconds per
    # launch, which only this 13-us kernel's figure carries).
    def back_to_back_ms(fn):
        for _ in range(3):
            fn()
        out = []
        for _ in range(3):
            ev[0].record(stream)
            for _ in range(args.steps):
                fn()
            ev[1].record(stream)
            torch.cuda.synchronize()
            out.append(ev[0].elapsed_time(ev[1]) / args.steps)
        return sorted(out)[1]

    def fwd_only():
        if fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), B, H, N, D,
               scale, causal, sp) != 0:
            raise RuntimeError("forward failed")

    def bwd_only():
        if bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(),
               do.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), B, H, N, D, scale,
               causal, sp) != 0:
            raise RuntimeError("backward failed")

    fwd_region = back_to_back_ms(fwd_only)
    bwd_region = back_to_back_ms(bwd_only)
    lib.profile_enable(True)
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    kernels = lib.profile_report()
    lib.profile_enable(False)

    f_fwd = flops_fwd(B, H, N, D, causal)
    f_bwd = 2.5 * f_fwd
    value = (f_fwd + f_bwd) / (ms_per_step * 1e-3) / 1e12

    # Algorithmic FLOPs per launch: forward = F_fwd; F_bwd counts five N^2 products (S, dP, dV,
    # dK, dQ). The backward runs its dkdv part (S, dP, dV, dK: 4/5 of F_bwd) and its dq part (dQ:
    # 1/5, plus a recompute of S and dP that the algorithmic count does not include) either in
    # one launch (backward_dq_dkdv, head_dim 128) or as two kernels.
    alg = {"forward": f_fwd, "backward_dq_dkdv": f_bwd, "backward_dq": f_bwd / 5,
           "backward_dkdv": f_bwd * 4 / 5}
    suffix = f"_bf16_d{D}"
    k_ms_hook = {label[:-len(suffix)]: tot / n for label, (n, tot) in kernels.items()
                 if label.endswith(suffix) and n}
    # Per-launch times from the back-to-back regions (the hook's figure beside each).
    k_ms = dict(k_ms_hook)
    method = {}
    if "forward" in k_ms:
        k_ms["forward"] = fwd_region
        method["forward"] = "back-to-back forward calls between two events"
    others = sum(v2 for k2, v2 in k_ms_hook.items()
                 if k2.startswith("backward") and k2 != "backward_dq_dkdv")
    if "backward_dq_dkdv" in k_ms:
        k_ms["backward_dq_dkdv"] = bwd_region - others
        method["backward_dq_dkdv"] = ("back-to-back backward calls between two events, minus "
                                      "the delta kernel's per-launch hook time")
    rooflines = []
    for name, flop in alg.items():
        if name not in k_ms:
            continue
        ms = k_ms[name]
        ach = flop / (ms * 1e-3) / 1e12
        rooflines.append({"kernel": name + suffix, "bound": "mfma", "achieved": round(ach, 2),
                          "peak": PEAK_BF16_TFLOPS, "unit": "TFLOP/s",
                          "frac": round(ach / PEAK_BF16_TFLOPS, 4), "avg_ms": round(ms, 4),
                          "avg_ms_event_pairs": round(k_ms_hook[name], 4),
                          "timing": method.get(name, "per-launch event hook"),
                          "alg_flop_per_launch": flop})
    dominant = max(rooflines, key=lambda r: r["avg_ms"])
    roofline = {k2: dominant[k2] for k2 in ("bound", "achieved", "peak", "unit", "frac")}
    roofline["traffic"] = committed_traffic(dominant["kernel"])
    roofline["traffic_source"] = (
        "not measured in this run: the rocprofv3 FETCH_SIZE / WRITE_SIZE figure committed in "
        "profiles/hbm_traffic_pmc.md for this kernel (bytes per launch; its range over runs is "
        "listed there)")
    roofline["kernel"] = dominant["kernel"]
    roofline["avg_ms"] = dominant["avg_ms"]
    roofline["timing"] = dominant["timing"]

    # ---------------- bounded parity check on the timed data ----------------
    parity = None
    if not args.no_parity:
        import oracle

        log("parity check (2 heads, oracle)")
        heads = [(0, 0), (B - 1, H - 1)]
        o_np, l_np = synth.to_numpy(o), synth.to_numpy(lse)
        dq_np, dk_np, dv_np = (synth.to_numpy(t) for t in (dq, dk, dv))
        errs = {"O": 0.0, "L": 0.0, "dQ": 0.0, "dK": 0.0, "dV": 0.0}
        rows = np.arange(0, N, 61, dtype=np.int64)
        for (b, h) in heads:
            sl = (slice(b, b + 1), slice(h, h + 1))
            qh, kh, vh, doh = (x[sl] for x in host)
            o_ref, l_ref = oracle.forward(qh, kh, vh, scale, causal, nthreads=host_threads())
            errs["O"] = max(errs["O"], float(np.abs(o_np[sl] - o_ref).max()))
            errs["L"] = max(errs["L"], float(np.abs(l_np[sl] - l_ref).max()))
            rq, rk, rv = oracle.backward_rows(qh, kh, vh, doh, scale, causal, rows, rows,
                                              nthreads=host_threads())
            errs["dQ"] = max(errs["dQ"], float(np.abs(dq_np[sl][:, :, rows] - rq).max()))
            errs["dK"] = max(errs["dK"], float(np.abs(dk_np[sl][:, :, rows] - rk).max()))
            errs["dV"] = max(errs["dV"], float(np.abs(dv_np[sl][:, :, rows] - rv).max()))
        parity = {"max_abs_err": {k2: round(v2, 6) for k2, v2 in errs.items()}, "tol": 2e-2,
                  "pass": all(v2 <= 2e-2 for v2 in errs.values()),
                  "sample": f"heads {heads}, O/L all rows, grads every 61st row"}

    del q, k, v, do, o, dq, dk, dv
    torch.cuda.empty_cache()

    # ---------------- extended entry points ----------------
    ext = None
    if not args.no_ext:
        log("extended forward / backward workloads")
        ext = bench_ext(lib, torch, max(3, args.steps // 4), stream)

    # ---------------- configs 1, 2 and 5 ----------------
    configs = None
    if not args.no_configs:
        log("configurations 1, 2 and 5")
        configs = bench_configs(lib, torch, max(3, args.steps // 4), stream)

    # ---------------- config 4: split-KV decode ----------------
    decode = None
    if not args.no_decode:
        Bd, Hd, LKV, Dd = CFG4["B"], CFG4["H"], CFG4["LKV"], CFG4["D"]
        log("generating config-4 inputs (torch generator on the GPU)")
        g = torch.Generator(device=dev)
        g.manual_seed(1)
        qd = torch.randn((Bd, Hd, 1, Dd), generator=g, device=dev, dtype=torch.float32).half()
        g.manual_seed(2)
        kd = torch.randn((Bd, Hd, LKV, Dd), generator=g, device=dev, dtype=torch.float16)
        g.manual_seed(3)
        vd = torch.randn((Bd, Hd, LKV, Dd), generator=g, device=dev, dtype=torch.float16)
        od = torch.empty_like(qd)
        ld = torch.empty((Bd, Hd, 1), device=dev, dtype=torch.float32)
        dec = lib.fn("decode", "f16")
        nbytes = decode_bytes(Bd, Hd, LKV, Dd)

        def time_calls(fn):
            """ms per call: the median of 5 regions of args.steps calls with no event hook (the
            hook's events between the split and combine launches cost time of their own), then
            the per-kernel report of a further pass with the hook on."""
            for _ in range(3):
                fn()
            torch.cuda.synchronize()
            regions = []
            for _ in range(5):
                t0.record(stream)
                for _ in range(args.steps):
                    fn()
                t1.record(stream)
                torch.cuda.synchronize()
                regions.append(t0.elapsed_time(t1) / args.steps)
            ms = sorted(regions)[len(regions) // 2]
            lib.profile_enable(True)
            for _ in range(args.steps):
                fn()
            torch.cuda.synchronize()
            rep = lib.profile_report()
            lib.profile_enable(False)
            return ms, rep
        results = {}
        for splits in (16, 32, 64, 0):
            def run():
                st = dec(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), od.data_ptr(),
                         ld.data_ptr(), Bd, Hd, LKV, Dd, Dd ** -0.5, splits, sp)
                if st != 0:
                    raise RuntimeError(f"decode status {st}")
            ms, rep = time_calls(run)
            split_ms = rep.get(f"decode_split_f16_d{Dd}", (1, float("nan")))
            results["auto" if splits == 0 else str(splits)] = {
                "ms": round(ms, 4), "GB/s": round(nbytes / (ms * 1e-3) / 1e9, 1),
                "split_kernel_ms": round(split_ms[1] / split_ms[0], 4)}
        # Config 4 asks for 16-64 chunks: the headline is the best of those. The automatic
        # choice (4 splits at this shape) lies outside that range and is reported beside it.
        in_range = {kk: vv for kk, vv in results.items() if kk != "auto"}
        best = max(in_range.items(), key=lambda kv: kv[1]["GB/s"])
        split_kernel_gbs = nbytes / (best[1]["split_kernel_ms"] * 1e-3) / 1e9
        decode = {"metric": "decode HBM GB/s (fp16, B=16 H=32 Lkv=32768 D=128)",
                  "value": best[1]["GB/s"], "unit": "GB/s", "best_splits": best[0],
                  "headline_splits": "best of 16, 32, 64 (config 4's range)",
                  "auto_splits_outside_config_range": results["auto"],
                  "by_splits": results, "alg_bytes": nbytes,
                  "roofline": {"bound": "hbm", "kernel": f"decode_split_f16_d{Dd}",
                               "achieved": round(split_kernel_gbs, 1), "peak": PEAK_HBM_GBS,
                               "unit": "GB/s", "frac": round(split_kernel_gbs / PEAK_HBM_GBS, 4),
                               "traffic": committed_traffic(f"decode_split_f16_d{Dd}")}}
        del kd, vd

        # Decode extensions at the config-4 size: grouped-query heads (32 query heads over 8
        # key/value heads, so each K/V row serves 4 query heads) and the same keys in a paged
        # cache (16-key pages in shuffled order). Reported beside the headline, not in `value`.
        Hkv, page = 8, 16
        torch.cuda.empty_cache()
        g.manual_seed(4)
        kg = torch.randn((Bd, Hkv, LKV, Dd), generator=g, device=dev, dtype=torch.float16)
        g.manual_seed(5)
        vg = torch.randn((Bd, Hkv, LKV, Dd), generator=g, device=dev, dtype=torch.float16)
        ext_bytes = Bd * Hkv * LKV * Dd * 2 * 2 + Bd * Hd * Dd * 2 * 2 + Bd * Hd * 4

        def time_ext(fn, label):
            ms, rep = time_calls(fn)
            sk = rep.get(f"decode_split_f16_d{Dd}", (1, float("nan")))
            return {"ms": round(ms, 4), "GB/s": round(ext_bytes / (ms * 1e-3) / 1e9, 1),
                    "split_kernel_ms": round(sk[1] / sk[0], 4),
                    "frac_of_hbm": round(ext_bytes / (ms * 1e-3) / 1e9 / PEAK_HBM_GBS, 4),
                    "alg_bytes": ext_bytes, "workload": label}

        gqa = lib.fn("decode_gqa", "f16")

        def run_gqa():
            st = gqa(qd.data_ptr(), kg.data_ptr(), vg.data_ptr(), od.data_ptr(), ld.data_ptr(),
                     Bd, Hd, Hkv, LKV, Dd, Dd ** -0.5, 0, sp)
            if st != 0:
                raise RuntimeError(f"decode_gqa status {st}")
        dext = {"gqa": time_ext(run_gqa, f"fp16 B={Bd} H={Hd} Hkv={Hkv} Lkv={LKV} D={Dd}")}

        npages = Bd * LKV // page
        kp = kg.reshape(Bd, Hkv, LKV // page, page, Dd).permute(0, 2, 3, 1, 4).reshape(
            npages, page, Hkv, Dd)
        vp = vg.reshape(Bd, Hkv, LKV // page, page, Dd).permute(0, 2, 3, 1, 4).reshape(
            npages, page, Hkv, Dd)
        del kg, vg
        perm = torch.randperm(npages, generator=g, device=dev)
        kp = kp[perm].contiguous()
        vp = vp[perm].contiguous()
        table = torch.argsort(perm).to(torch.int32).reshape(Bd, LKV // page).contiguous()
        lens = torch.full((Bd,), LKV, dtype=torch.int32, device=dev)
        paged = lib.fn("decode_paged", "f16")

        def run_paged():
            st = paged(qd.data_ptr(), kp.data_ptr(), vp.data_ptr(), od.data_ptr(), ld.data_ptr(),
                       table.data_ptr(), lens.data_ptr(), Bd, Hd, Hkv, page, LKV // page, Dd,
                       Dd ** -0.5, 0, sp)
            if st != 0:
                raise RuntimeError(f"decode_paged status {st}")
        dext["paged"] = time_ext(run_paged, f"fp16 B={Bd} H={Hd} Hkv={Hkv} Lkv={LKV} D={Dd}, "
                                           f"{page}-key pages in shuffled order")
        decode["extensions"] = dext
        del kp, vp, table, lens, perm

    # ---------------- informational comparisons (after every measured record) ----------
    # A failure in one of them is recorded in its place and does not cost the JSON line.
    def informational(label, fn):
        log(label)
        try:
            return fn()
        except Exception as e:  # noqa: BLE001 - reported, never the headline
            torch.cuda.synchronize()
            return {"error": f"{type(e).__name__}: {str(e)[:200]}"}

    reference_shapes = None
    if not args.no_reference_shapes:
        reference_shapes = informational(
            "the reference's published timing shapes",
            lambda: bench_reference_shapes(torch, max(3, args.steps // 10)))

    sdpa = None
    if not args.no_sdpa:
        sdpa = informational(
            "torch scaled_dot_product_attention (fused kernels) beside this library",
            lambda: bench_sdpa(torch, max(5, args.steps // 5)))

    decode_graph = None
    if not args.no_decode_graph:
        decode_graph = informational(
            "decode calls eager and from a captured graph",
            lambda: bench_decode_graph(lib, torch, max(5, args.steps // 5)))

    # ---------------- CPU baseline (bounded sample) ----------------
    cpu = None
    if not args.no_cpu_baseline:
        cpu = cpu_baseline(host, B, H, N, D, scale, causal, args.cpu_seconds,
                           with_decode=not args.no_decode)

    out = {
        "metric": "fwd+bwd TFLOP/s (bf16 causal N=4096 D=128) + decode HBM GB/s at 32k KV",
        "value": round(value, 2),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ramp": {"ms": args.ramp_ms, "steps": ramp_steps},
        "ms_per_step": round(ms_per_step, 4),
        "timing": {"regions": nreg, "steps_per_region": sizes,
                   "region_ms_per_step": [round(x, 4) for x in region_ms],
                   "ms_per_step_mean": round(ms_per_step_mean, 4),
                   "headline": "median over the regions"},
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (SplitMix64/Box-Muller N(0,1), seeds 1-4; decode: torch GPU generator)",
        "config": {"workload": "cfg3 fwd+bwd: bf16 causal B=2 H=16 N=4096 D=128 (one step = one "
                               "forward + one backward); cfg4 decode reported under 'decode'",
                   "batch": B, "heads": H, "seq_len": N, "head_dim": D, "causal": causal},
        "fwd_ms": round(k_ms["forward"], 4),
        "bwd_ms": round(sum(v2 for k2, v2 in k_ms.items() if k2.startswith("backward")), 4),
        "roofline": roofline,
        "rooflines": rooflines,
        "kernel_ms": {kk: round(vv, 4) for kk, vv in k_ms.items()},
        "decode": decode,
        "ext": ext,
        "sdpa": sdpa,
        "reference_shapes": reference_shapes,
        "decode_graph": decode_graph,
        "configs": configs,
        "parity": parity,
        "cpu_baseline": cpu,
    }
    if cpu:
        # Same problem on both sides: config 3's fwd + bwd (and config 4's decode bytes).
        out["cpu_baseline"]["gpu_speedup"] = round(value / cpu["value"], 1)
        if decode and "decode" in cpu:
            cpu["decode"]["gpu_speedup"] = round(decode["value"] / cpu["decode"]["value"], 1)
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
