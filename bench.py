"""Benchmark of the MI355X quantized-KV attention path (one JSON line on stdout).

Headline workload: FP8-E4M3 KV-cache flash-decode, batch 32,
32 query / 8 KV heads, head_dim 128, every sequence at context 8192, bf16 queries and outputs;
cached K/V from bf16 N(0,1) with 1 % of channels x8, per-(token, head) absmax/448 scales.
A step is one decode call over the whole batch with the cache resident in HBM. At this shape the
split rule picks one split, so one call is one launch of the decode kernel (no combine pass).
Two cache copies (554 MB each, both larger than the 256 MB MALL) are used alternately so every
call streams from HBM.

value = algorithmic HBM bytes per call (codes + scales + q + out) / measured seconds per call,
timed with HIP events on the stream the library launches on (torch's current stream);
roofline.achieved = the same bytes / the decode kernel's average duration (the same figure, as
one call is one launch). roofline.traffic = HBM bytes per launch read by rocprofv3's FETCH_SIZE
and WRITE_SIZE counters, scaled by what they read for a plain copy of known size; it is taken
from the committed counter summary only while that summary's kernel-source digest equals these
sources' (csrc_digest), and is null otherwise. cpu_baseline = the oracle's
restatement of the reference CPU path (dequantize -> bf16 -> f32 unfused attention), timed on the
host on a bounded sample of the same workload.

"other_configs" reports BASELINE configs 3 (MXFP4, ragged), 4 (causal bf16 prefill with fused
FP8 append) and 5 (TurboQuant-4, context 128K) with the same timing method; they are secondary
figures, not the headline value. "c2_shape_mxfp8" / "c2_shape_nvfp4" time the decode of the
other block-scaled formats at the config-2 shape; "c4_shape_fp8_kv" the attention over E4M3
K / V with descales at the config-4 shape; "ra_*" time the fused RoPE + FP8
quantize-append at the config-4 prefill shape and at one config-2 decode step; "append_c2_shape"
the plain quantize-and-append of each format and side.
Each "cpu_baseline" is the oracle's restatement of the reference CPU path, timed on this host's
CPUs (all of those this process may use) on a bounded sample of the workload and scaled to it.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu] [--no-extra]
                       [--only c2,c3,c4,c5,tp,f8,fx,ap,ra,pd,pp,fq] [--calibration-copy]
"""
from __future__ import annotations

import argparse
import json
import os
import re
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
BF16_PEAK_TFLOPS = 2516.6
TRAFFIC_SUMMARY = os.path.join(ROOT, "profiles", "decode_fp8_c2_and_append_rows_traffic.md")


def load_cqkv():
    import importlib.util
    spec = importlib.util.spec_from_file_location(
        "cqkv", os.path.join(ROOT, "candle-rocm-vulkan_amd", "cqkv.py"))
    mod = importlib.util.module_from_spec(spec)
    sys.modules["cqkv"] = mod
    spec.loader.exec_module(mod)
    return mod


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def kv_gpu(shape, seed, dev, outliers=True):
    import torch
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(*shape, generator=g, device=dev)
    if outliers:
        mask = torch.rand(shape[1], shape[3], generator=g, device=dev) < 0.01
        x = torch.where(mask[None, :, None, :], x * 8.0, x)
    return x.to(torch.bfloat16)


def build_cache(cq, fmt, b, hkv, d, ctx, dev, seed, chunk=2048, vfmt=None):
    cache = cq.TurboKvCache(fmt, fmt if vfmt is None else vfmt, b, hkv, d, ctx, device=dev)
    for t0 in range(0, ctx, chunk):
        t = min(chunk, ctx - t0)
        cache.append(kv_gpu((b, hkv, t, d), seed + t0, dev),
                     kv_gpu((b, hkv, t, d), seed + 7 + t0, dev))
    return cache


LAST_MEDIAN_MS = [0.0]  # median per-call time of the last time_calls


def time_calls(fn, steps, warmup, stream):
    """Mean ms per call over exactly `steps` back-to-back calls after `warmup` untimed ones,
    between two HIP events on the library's stream. A second pass of `steps` calls with an event
    after each call gives the per-call times, whose median goes to LAST_MEDIAN_MS (kept apart
    from the first pass, whose calls run back to back with no event between them)."""
    import torch
    for i in range(warmup):
        fn(i)
    torch.cuda.synchronize()
    start = torch.cuda.Event(enable_timing=True)
    stop = torch.cuda.Event(enable_timing=True)
    start.record(stream)
    for i in range(steps):
        fn(i)
    stop.record(stream)
    torch.cuda.synchronize()
    mean = start.elapsed_time(stop) / steps
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(steps + 1)]
    ev[0].record(stream)
    for i in range(steps):
        fn(i)
        ev[i + 1].record(stream)
    torch.cuda.synchronize()
    per = sorted(ev[i].elapsed_time(ev[i + 1]) for i in range(steps))
    LAST_MEDIAN_MS[0] = per[len(per) // 2] if len(per) % 2 else 0.5 * (per[len(per) // 2 - 1] +
                                                                         per[len(per) // 2])
    return mean  # ms per call


def row_bytes(fmt, d):
    """Packed cache bytes of one (token, head) row: codes + its scales."""
    return {5: d + 4, 2: d // 2 + d // 32, 0: d // 2 + 4, 4: d + d // 32,
            3: d // 2 + d // 16 + 4, 1: d // 2 + 8 + d // 8}[fmt]


def decode_bytes(b, hq, hkv, d, total_tokens, fmt, vfmt=None):
    """K + V rows over `total_tokens` (summed over the batch) for every kv head, plus q and out."""
    vfmt = fmt if vfmt is None else vfmt
    return (hkv * total_tokens * (row_bytes(fmt, d) + row_bytes(vfmt, d))
            + 2 * b * hq * d * 2)


def csrc_digest() -> str:
    """sha256 over the library's kernel sources (csrc/*.hip, *.h, *.cpp and include/cqkv.h, in
    name order): the counter summaries record the digest of the sources they were taken from."""
    import hashlib
    h = hashlib.sha256()
    src = os.path.join(ROOT, "candle-rocm-vulkan_amd", "csrc")
    files = sorted(f for f in os.listdir(src) if f.endswith((".hip", ".h", ".cpp")))
    for name in files + ["../../include/cqkv.h"]:
        with open(os.path.join(src, name), "rb") as f:
            h.update(os.path.basename(name).encode() + b"\0" + f.read())
    return h.hexdigest()


def read_traffic():
    """HBM bytes per decode launch from the committed counter summary, or None when the summary
    is missing or was taken from other kernel sources than these (csrc_digest)."""
    try:
        with open(TRAFFIC_SUMMARY) as f:
            text = f.read()
    except OSError:
        return None
    m = re.search(r"traffic_bytes_per_launch:\s*([0-9]+)", text)
    d = re.search(r"csrc_sha256:\s*([0-9a-f]{64})", text)
    if not m or not d or d.group(1) != csrc_digest():
        return None
    return int(m.group(1))


def cpu_info():
    """Threads the CPU baseline uses (every CPU this process may run on), the machine's logical
    CPU count and model."""
    threads = len(os.sched_getaffinity(0))
    model = "unknown"
    try:
        with open("/proc/cpuinfo") as f:
            for line in f:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    return threads, {"nproc": os.cpu_count(), "cpu_model": model}


def side_rows(cq, side, b0, nb, tokens):
    """Reference rows (nb, kv_heads, tokens, words) of sequences b0 .. b0 + nb - 1 of a cache side
    (its planes are batch-major, so those sequences are one contiguous slice)."""
    import numpy as np
    cb, sb = side.codes.numel() // side.batch, side.scales.numel() // side.batch
    view = cq.CacheSide(side.fmt, side.is_value, nb, side.kv_heads, side.head_dim, side.capacity,
                        side.codes[b0 * cb:(b0 + nb) * cb], side.scales[b0 * sb:(b0 + nb) * sb],
                        side.seed, side.rotation, side.qjl, side.bits, side.rot)
    return cq.rows_export(view, tokens).cpu().numpy().view(np.uint32)


def timed_reps(fn, budget_s=10.0, max_reps=20):
    reps, t_total = 0, 0.0
    while t_total < budget_s and reps < max_reps:
        t0 = time.perf_counter()
        fn()
        t_total += time.perf_counter() - t0
        reps += 1
    return t_total / reps, reps


def cpu_baseline_decode(cq, cache, q, fmt, seqs, tokens, scale, threads, kv_lens=None,
                        vfmt=None):
    """The oracle's restatement of the reference CPU decode path (dequantize, unrotate, bf16
    cache, unfused f32 attention) over the sequences `seqs` (a contiguous range); returns seconds
    for that sample and the repetitions timed."""
    import numpy as np
    from oracle import oracle as O
    vfmt = fmt if vfmt is None else vfmt
    b0, nb = seqs[0], len(seqs)
    kr = side_rows(cq, cache.k, b0, nb, tokens)
    vr = side_rows(cq, cache.v, b0, nb, tokens)
    qb = O.f32_to_bf16_bits(q[b0:b0 + nb].float().cpu().numpy())
    turbo = (O.TURBO_MSE, O.TURBO_PROD)
    bits = {f: (4 if f in turbo else 0) for f in (fmt, vfmt)}
    d = q.shape[-1]
    pk = O.rotation_matrix(d, O.ROT_HADAMARD, cache.k.seed) if fmt in turbo else None
    pv = O.rotation_matrix(d, O.ROT_HADAMARD, cache.v.seed) if vfmt in turbo else None
    sk = O.qjl_matrix(d, cache.k.seed) if fmt == O.TURBO_PROD else None
    lens = None if kv_lens is None else np.array(kv_lens[b0:b0 + nb], np.int32)
    return timed_reps(lambda: O.cache_attention(qb, kr, vr, (fmt, bits[fmt]), (vfmt, bits[vfmt]),
                                                pk, pv, tokens, scale, kv_lens=lens,
                                                threads=threads, qjl_k=sk))


def cpu_baseline_prefill(threads, heads=4):
    """Config 4 on the CPU: the oracle's causal f32 attention (the reference's unfused CPU path)
    for `heads` query heads (one kv head) of one sequence, plus the FP8 quantize_rows of that
    sequence's K / V rows; returns seconds scaled to the whole call (4 sequences x 32 heads)."""
    import numpy as np
    from oracle import oracle as O
    s, d = 4096, 128
    rng = np.random.default_rng(7)
    q = O.round_bf16(rng.standard_normal((1, heads, s, d), dtype=np.float32))
    k = O.round_bf16(rng.standard_normal((1, 1, s, d), dtype=np.float32))
    v = O.round_bf16(rng.standard_normal((1, 1, s, d), dtype=np.float32))
    kv_rows = O.round_bf16(rng.standard_normal((8 * s, d), dtype=np.float32))
    t_att, reps = timed_reps(lambda: O.attention_unfused(q, k, v, 1.0 / d ** 0.5, wl=-1, wr=0,
                                                         threads=threads), max_reps=5)
    t_app, _ = timed_reps(lambda: (O.quantize_rows(O.FP8, 0, kv_rows, threads=threads),
                                   O.quantize_rows(O.FP8, 0, kv_rows, threads=threads)),
                          budget_s=2.0, max_reps=5)
    return t_att * (4 * 32 / heads) + t_app * 4, reps, heads


def cpu_baseline_entry(value, unit, us_per_call, threads, info, sample, reps):
    e = {"value": value, "unit": unit, "cores": threads, "kind": "port",
         "us_per_call": round(us_per_call, 1), "reps": reps,
         "sample": sample}
    e.update(info)
    return e


def decode_case(cq, dev, stream, fmt, b, hq, hkv, d, ctx, steps, warmup, lens=None, chunk=2048,
                vfmt=None):
    """Build two cache copies, time `steps` decode calls alternating between them."""
    import torch
    scale = 1.0 / d ** 0.5
    caches = [build_cache(cq, fmt, b, hkv, d, ctx, dev, 1000 * i + 11 * fmt, chunk, vfmt)
              for i in range(2)]
    q = kv_gpu((b, hq, 1, d), 5, dev, outliers=False)
    out = torch.empty_like(q)
    kv_lens = None if lens is None else torch.tensor(lens, dtype=torch.int32, device=dev)
    # workspace for the split count the call will pick, so no call allocates inside the timing
    splits = cq.decode_splits(b, hkv, ctx, fmt, ragged=lens is not None,
                              v_fmt=fmt if vfmt is None else vfmt)
    ws = torch.zeros(max(1, cq.decode_workspace_bytes(b, hq, 1, d, splits)), dtype=torch.uint8,
                     device=dev)

    def step(i):
        c = caches[i & 1]
        cq.decode_attention(q, c.k, c.v, ctx, scale, kv_lens=kv_lens, out=out, splits=0,
                            workspace=ws)

    ms = time_calls(step, steps, warmup, stream)
    total = b * ctx if lens is None else int(sum(lens))
    nbytes = decode_bytes(b, hq, hkv, d, total, fmt, vfmt)
    return caches, q, ms, nbytes


def prefill_case(cq, dev, stream, steps, warmup):
    """causal bf16 prefill, B=4, S=4096, 32/8 heads, d=128, fused FP8
    append of K and V into a cache."""
    import torch
    b, s, hq, hkv, d = 4, 4096, 32, 8, 128
    g = torch.Generator(device=dev).manual_seed(7)
    q = torch.randn(b, s, hq, d, generator=g, device=dev).to(torch.bfloat16)
    k = torch.randn(b, s, hkv, d, generator=g, device=dev).to(torch.bfloat16)
    v = torch.randn(b, s, hkv, d, generator=g, device=dev).to(torch.bfloat16)
    out = torch.empty_like(q)
    kc = cq.CacheSide.empty(cq.FP8, False, b, hkv, d, s, dev)
    vc = cq.CacheSide.empty(cq.FP8, True, b, hkv, d, s, dev)

    def step(i):
        cq.flash_attn(q, k, v, 1.0 / d ** 0.5, True, out=out, k_cache=kc, v_cache=vc)

    ms = time_calls(step, steps, warmup, stream)
    flops = 2 * b * hq * s * s * d  # causal: half of 4*B*H*S^2*D
    tflops = flops / (ms * 1e-3) / 1e12
    return {"workload": "BASELINE config 4: causal bf16 prefill + fused FP8 K/V append",
            "batch": b, "seq_len": s, "q_heads": hq, "kv_heads": hkv, "head_dim": d,
            "us_per_call": round(ms * 1e3, 2),
            "median_us_per_call": round(LAST_MEDIAN_MS[0] * 1e3, 2), "flop_per_call": flops,
            "achieved_tflops": round(tflops, 1), "peak_tflops": BF16_PEAK_TFLOPS,
            "frac": round(tflops / BF16_PEAK_TFLOPS, 4), "bound": "mfma",
            "timed": "whole call: pre-pass (V transpose + fused FP8 K/V append) + prefill kernel"}


def rope_append_case(cq, dev, stream, fmt, b, hq, hkv, d, t, cap, steps, warmup):
    """Fused RoPE + quantize-append from a (b, t, (hq + 2 hkv) d) bf16 QKV projection output:
    rotated q written out (bf16), K rotated and V quantized into the cache at position 0."""
    import torch
    qkv = kv_gpu((b, t, 1, (hq + 2 * hkv) * d), 17, dev)[:, :, 0].contiguous()
    q, k, v = cq.split_qkv(qkv, hq, hkv)
    ang = torch.arange(cap, dtype=torch.float64, device=dev)[:, None] / \
        10000.0 ** (torch.arange(0, d, 2, dtype=torch.float64, device=dev) / d)
    cos, sin = ang.cos().to(torch.bfloat16), ang.sin().to(torch.bfloat16)
    ks = cq.CacheSide.empty(fmt, False, b, hkv, d, cap, dev)
    vs = cq.CacheSide.empty(fmt, True, b, hkv, d, cap, dev)
    q_out = torch.empty(b, hq, t, d, dtype=torch.bfloat16, device=dev)

    def call():
        cq.rope_quant_append(ks, vs, q, k, v, cos, sin, cq.ROPE_HALVES, 0, q_out=q_out)
    timed = "one cqkv_rope_quant_append launch"
    if t > 1:
        ms = time_calls(lambda i: call(), steps, warmup, stream)
    else:
        # one decode step is a few microseconds of GPU work, less than the Python call: replay a
        # captured HIP graph of `reps` calls so the figure is the GPU's (the path records no
        # memset node; every replay is checked against the eager result by the tests' rule)
        reps = 20
        call()
        torch.cuda.synchronize()
        want = q_out.clone()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for _ in range(reps):
                call()
        g.replay()
        torch.cuda.synchronize()
        if not torch.equal(q_out, want):
            raise RuntimeError("graph replay of the fused RoPE + append differs from eager")
        ms = time_calls(lambda i: g.replay(), max(5, steps // reps), 2, stream) / reps
        timed = f"one launch; a HIP graph of {reps} captured calls replayed"
    rb = row_bytes(fmt, d)
    nbytes = (qkv.numel() * 2 + 2 * t * (d // 2) * 2 + q_out.numel() * 2
              + 2 * b * hkv * t * rb)
    gbs = nbytes / (ms * 1e-3) / 1e9
    return {"workload": f"fused RoPE + {['TURBO4', '', 'MXFP4', 'NVFP4', 'MXFP8', 'FP8'][fmt]} append, "
                        f"B={b} t={t} Hq={hq} Hkv={hkv} D={d}",
            "us_per_call": round(ms * 1e3, 2), "bytes_per_call": nbytes,
            "roofline": {"bound": "hbm", "achieved": round(gbs, 1), "peak": HBM_PEAK_GBS,
                         "unit": "GB/s", "frac": round(gbs / HBM_PEAK_GBS, 4)},
            "timed": timed}


def fp8_attn_case(cq, dev, stream, steps, warmup):
    """Causal attention over E4M3 K / V with per-tensor descales (flash_attn_fp8's attention):
    the E4M3 -> bf16 staging pass plus the MFMA prefill, B=4 S=4096 32/8 heads D=128."""
    import torch
    B, S, HQ, HKV, D = 4, 4096, 32, 8, 128
    q = kv_gpu((B, S, HQ, D), 41, dev, outliers=False)
    k = kv_gpu((B, S, HKV, D), 42, dev)
    v = kv_gpu((B, S, HKV, D), 43, dev)
    k8, ks = cq.fp8_quantize_tensor(k)
    v8, vs = cq.fp8_quantize_tensor(v)
    out = torch.empty_like(q)

    def step(i):
        cq.flash_attn_fp8_codes(q, k8, v8, 1.0 / D ** 0.5, True, 1.0, 1.0, k_scale=ks,
                                v_scale=vs, out=out)
    ms = time_calls(step, steps, warmup, stream)
    flops = 2 * B * HQ * S * S * D
    return {"workload": "FP8 (E4M3) K / V causal attention with descales, config-4 shape",
            "us_per_call": round(ms * 1e3, 2), "flop_per_call": flops,
            "achieved_tflops": round(flops / (ms * 1e-3) / 1e12, 1),
            "peak_tflops": BF16_PEAK_TFLOPS,
            "frac": round(flops / (ms * 1e-3) / 1e12 / BF16_PEAK_TFLOPS, 4), "bound": "mfma",
            "timed": "whole call: E4M3 -> bf16 staging, V transpose pre-pass, prefill kernel"}


def plain_decode_case(cq, dev, stream, steps, warmup, dtype, B=32, HQ=32, HKV=8, D=128,
                      CTX=8192, q_dtype=None):
    """flash_attn over plain K / V at the config-2 decode shape (one query per sequence): the
    split-K row kernel (f32 queries: the f32 kernel); bytes = the K and V rows read (the queries
    and outputs are 0.02 %)."""
    import torch
    q_dtype = q_dtype or dtype
    q = kv_gpu((B, 1, HQ, D), 61, dev, outliers=False).to(q_dtype)
    k = kv_gpu((B, CTX, HKV, D), 62, dev).to(dtype)
    v = kv_gpu((B, CTX, HKV, D), 63, dev).to(dtype)
    out = torch.empty_like(q)
    ws = torch.empty(max(cq.flash_attn_workspace_bytes(q_dtype, B, 1, CTX, HQ, HKV, D), 1),
                     dtype=torch.uint8, device=dev)
    ms = time_calls(lambda i: cq.flash_attn(q, k, v, 1.0 / D ** 0.5, True, out=out,
                                            workspace=ws), steps, warmup, stream)
    nbytes = 2 * B * CTX * HKV * D * k.element_size()
    del q, k, v
    torch.cuda.empty_cache()
    qn = "" if q_dtype == dtype else f"{str(q_dtype)[6:]} queries, "
    return decode_summary(f"flash_attn decode, {qn}plain {str(dtype)[6:]} K / V, config-2 shape",
                          ms, nbytes, {"batch": B, "q_heads": HQ, "kv_heads": HKV,
                                       "head_dim": D, "context": CTX,
                                       "timed": "whole call (split-K row kernel + combine)"})


def plain_prefill_case(cq, dev, stream, steps, warmup, dtype, D, B=4, S=4096, HQ=32, HKV=8,
                       q_dtype=None):
    """Causal flash_attn on the plain-dtype kernel (f16, or a head dim other than 128), or with
    f32 queries on split bf16 operands (roofline: the bf16 MFMA peak over its six products)."""
    import torch
    q_dtype = q_dtype or dtype
    q = kv_gpu((B, S, HQ, D), 71, dev, outliers=False).to(q_dtype)
    k = kv_gpu((B, S, HKV, D), 72, dev).to(dtype)
    v = kv_gpu((B, S, HKV, D), 73, dev).to(dtype)
    out = torch.empty_like(q)
    ws = torch.empty(max(cq.flash_attn_workspace_bytes(q_dtype, B, S, S, HQ, HKV, D), 1),
                     dtype=torch.uint8, device=dev)
    ms = time_calls(lambda i: cq.flash_attn(q, k, v, 1.0 / D ** 0.5, True, out=out,
                                            workspace=ws), steps, warmup, stream)
    flops = 2 * B * HQ * S * S * D  # causal: half of 4 B HQ S^2 D
    del q, k, v
    torch.cuda.empty_cache()
    tf = flops / (ms * 1e-3) / 1e12
    f32 = q_dtype == torch.float32
    # f32 queries: six bf16 products each (three exact bf16 parts per operand)
    peak = BF16_PEAK_TFLOPS / 6 if f32 else BF16_PEAK_TFLOPS
    kind = "f32 on split bf16 operands" if f32 else "plain-dtype kernel"
    qn = "" if q_dtype == dtype else f"{str(q_dtype)[6:]} queries over "
    return {"workload": f"causal flash_attn, {qn}{str(dtype)[6:]}, D={D}, B={B} S={S} "
                        f"{HQ}/{HKV} heads ({kind})",
            "us_per_call": round(ms * 1e3, 2), "flop_per_call": flops,
            "achieved_tflops": round(tf, 1), "peak_tflops": peak,
            "frac": round(tf / peak, 4), "bound": "mfma", "timed": "whole call"}


def append_case(cq, dev, stream, steps, warmup, b=32, hkv=8, d=128, t=2048):
    """cqkv_quant_append alone: B=32 sequences x 8 kv heads x 2048 tokens (524,288 rows of the
    config-2 cache shape) of bf16 K or V into FP8 / MXFP4 / TURBO4 / MXFP8 / NVFP4 sides (TurboProd: keys only) at
    position 0. Bytes = the bf16 rows read plus the codes and scales written."""
    import torch
    x = kv_gpu((b, hkv, t, d), 51, dev)
    res = {}
    names = {cq.FP8: "fp8", cq.MXFP4: "mxfp4", cq.TURBO4: "turbo4", cq.MXFP8: "mxfp8",
             cq.NVFP4: "nvfp4", cq.TURBOPROD: "turboprod"}
    for fmt, name in names.items():
        for is_value in ((False,) if fmt == cq.TURBOPROD else (False, True)):
            side = cq.CacheSide.empty(fmt, is_value, b, hkv, d, t, dev, seed=44 if is_value else 42)
            ms = time_calls(lambda i: cq.quant_append(side, x, 0), steps, warmup, stream)
            nbytes = x.numel() * 2 + b * hkv * t * row_bytes(fmt, d)
            gbs = nbytes / (ms * 1e-3) / 1e9
            res[f"{name}_{'values' if is_value else 'keys'}"] = {
                "us_per_call": round(ms * 1e3, 2), "bytes_per_call": nbytes,
                "achieved_gbs": round(gbs, 1), "frac": round(gbs / HBM_PEAK_GBS, 4)}
            del side
    torch.cuda.empty_cache()
    return {"workload": f"cqkv_quant_append of bf16 rows, B={b} x {hkv} kv heads x {t} tokens, "
                        f"D={d}", "bound": "hbm", "peak_gbs": HBM_PEAK_GBS,
            "timed": "one quant_append launch per call", "per_side": res}


def decode_summary(name, ms, nbytes, extra):
    gbs = nbytes / (ms * 1e-3) / 1e9
    res = {"workload": name, "us_per_call": round(ms * 1e3, 2),
           "median_us_per_call": round(LAST_MEDIAN_MS[0] * 1e3, 2), "bytes_per_call": nbytes,
           "achieved_gbs": round(gbs, 1), "peak_gbs": HBM_PEAK_GBS,
           "frac": round(gbs / HBM_PEAK_GBS, 4), "bound": "hbm"}
    res.update(extra)
    return res


def calibration_copy(dev, reps=3):
    """A plain device copy of 1 GiB, `reps` times: the counter scale of FETCH_SIZE/WRITE_SIZE."""
    import torch
    n = 1 << 30
    src = torch.ones(n, dtype=torch.uint8, device=dev)
    dst = torch.empty_like(src)
    for _ in range(reps):
        dst.copy_(src)
    torch.cuda.synchronize()
    log(f"calibration copy: {reps} x {n} bytes read and written")


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=100)
    # The part's clocks reach their steady state after ~50-100 ms of back-to-back decode calls:
    # with 20 untimed calls the headline decode timed 96 us per call, after ~600 calls 89.4 us.
    ap.add_argument("--warmup", type=int, default=1000)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-extra", action="store_true", help="headline workload only")
    ap.add_argument("--only", default="",
                    help="comma list of c2,c3,c4,c5,tp,f8,fx,ap,ra,pd,pp,fq (default: all)")
    ap.add_argument("--calibration-copy", action="store_true",
                    help="also run a plain 1 GiB copy (for counter scaling)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build runs on one GPU only (asked for --gpus {args.gpus}); "
              "the path would shard by sequence / kv head with no exchange between GPUs",
              file=sys.stderr)
        sys.exit(2)

    import torch
    cq = load_cqkv()
    cq.lib()
    threads, info = cpu_info()
    dev = torch.device("cuda:0")
    stream = torch.cuda.current_stream(dev)
    only = set(x for x in args.only.split(",") if x)
    want = (lambda c: c in only) if only else (lambda c: c == "c2" or not args.no_extra)
    if args.calibration_copy:
        calibration_copy(dev)

    res = None
    if want("c2"):
        B, HQ, HKV, D, CTX = 32, 32, 8, 128, 8192
        log("config 2: FP8 decode B=32 32/8 d=128 ctx 8192")
        caches, q, ms, nbytes = decode_case(cq, dev, stream, cq.FP8, B, HQ, HKV, D, CTX,
                                            args.steps, args.warmup)
        splits = cq.decode_splits(B, HKV, CTX)
        achieved = nbytes / (ms * 1e-3) / 1e9  # GB/s
        log(f"config 2: {ms * 1e3:.2f} us/call, {achieved:.1f} GB/s")
        cpu = None
        if not args.no_cpu:
            sec, reps = cpu_baseline_decode(cq, caches[0], q, cq.FP8, range(2), CTX,
                                            1.0 / D ** 0.5, threads)
            sec *= B / 2
            cpu = cpu_baseline_entry(
                round(nbytes / sec / 1e12, 6), "TB/s", sec * 1e6, threads, info,
                "oracle cache_attention (the reference CPU decode path restated in C: "
                "dequantize, bf16 cache, unfused f32 attention) on 2 of the 32 sequences, "
                "scaled x16 to the full call", reps)
            log(f"cpu baseline: {sec * 1e6:.0f} us/call on {threads} threads")
        del caches
        traffic = read_traffic()
        res = {
            "metric": "quant-KV flash-decode µs/call + achieved HBM TB/s; bf16 prefill TFLOP/s",
            "value": round(achieved / 1000.0, 4),
            "unit": "TB/s",
            "n_gpus": 1,
            "steps": args.steps,
            "warmup": args.warmup,
            "ms_per_step": round(ms, 5),
            "us_per_call": round(ms * 1e3, 2),
            "median_us_per_call": round(LAST_MEDIAN_MS[0] * 1e3, 2),
            "timing": "ms_per_step / us_per_call: HIP events on the library's stream around the "
                      "K back-to-back timed calls (their mean); median_us_per_call: the median "
                      "of K more calls with an event after each",
            "higher_is_better": True,
            "scaling": "weak",
            "vs_baseline": None,
            "dtype": "fp8-e4m3 cache codes, bf16 q/out, f32 accumulate",
            "data": "synthetic (torch N(0,1) bf16, 1% channels x8)",
            "config": {"workload": "BASELINE config 2: FP8-KV GQA flash-decode", "batch": B,
                       "q_heads": HQ, "kv_heads": HKV, "head_dim": D, "context": CTX,
                       "splits": splits, "cache_copies": 2, "parallelism": "single GPU"},
            "roofline": {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS,
                         "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 4),
                         "traffic": traffic, "bytes_per_call": nbytes,
                         "timed": "decode kernel (one launch per call at this shape)"},
            "cpu_baseline": cpu,
        }
        torch.cuda.empty_cache()

    other = {}
    steps_x = max(5, args.steps // 5)
    warm_x = max(2, args.warmup // 2)
    if want("c4"):
        # MFMA-bound: give the clocks time to settle after the HBM-bound decode workloads
        log("config 4: causal prefill + fused FP8 append")
        # the MFMA clocks settle over the first ~100 calls: a longer untimed warm-up
        other["c4_prefill"] = prefill_case(cq, dev, stream, max(steps_x, 20), max(warm_x, 80))
        log(f"config 4: {other['c4_prefill']['us_per_call']} us/call")
        if not args.no_cpu:
            sec, reps, heads = cpu_baseline_prefill(threads)
            other["c4_prefill"]["cpu_baseline"] = cpu_baseline_entry(
                round(other["c4_prefill"]["flop_per_call"] / sec / 1e12, 6), "TFLOP/s",
                sec * 1e6, threads, info,
                f"oracle attention_unfused (the reference CPU path: f32 q k^T, scale, mask, "
                f"softmax, p v) causal on {heads} of the 32 query heads of sequence 0, plus the "
                f"FP8 quantize_rows of its 8 x 4096 K and V rows, scaled to the 4 x 32 heads", reps)
            log(f"config 4 cpu: {sec * 1e6:.0f} us/call")
        torch.cuda.empty_cache()
    if want("c3"):
        import random
        rng = random.Random(3)
        lens = [rng.randint(1024, 32768) for _ in range(64)]
        log("config 3: MXFP4 ragged decode B=64 32/8 d=128")
        caches, q3, ms, nbytes = decode_case(cq, dev, stream, cq.MXFP4, 64, 32, 8, 128, 32768,
                                             steps_x, warm_x, lens=lens)
        other["c3_mxfp4_ragged"] = decode_summary(
            "BASELINE config 3: MXFP4-KV ragged decode", ms, nbytes,
            {"batch": 64, "q_heads": 32, "kv_heads": 8, "head_dim": 128,
             "lens": "uniform [1024, 32768], random.Random(3)", "sum_len": int(sum(lens)),
             "dtype": "e2m1 codes with e8m0 block scales; bf16 MFMA operands: keys exact, "
                      "bf16 queries exact, P times each key's value block scale as one bf16 "
                      "operand (8 significant bits); f32 accumulate",
             "timed": "whole call (split-K decode + combine)"})
        log(f"config 3: {ms * 1e3:.2f} us/call")
        if not args.no_cpu:
            sec, reps = cpu_baseline_decode(cq, caches[0], q3, cq.MXFP4, range(2), 32768,
                                            1.0 / 128 ** 0.5, threads, kv_lens=lens)
            sec *= sum(lens) / sum(lens[:2])  # the CPU path's work is linear in the keys
            other["c3_mxfp4_ragged"]["cpu_baseline"] = cpu_baseline_entry(
                round(nbytes / sec / 1e12, 6), "TB/s", sec * 1e6, threads, info,
                f"oracle cache_attention on sequences 0-1 ({lens[0] + lens[1]} keys), scaled by "
                f"the key count to the call's {sum(lens)}", reps)
            log(f"config 3 cpu: {sec * 1e6:.0f} us/call")
        del caches
        torch.cuda.empty_cache()
    if want("c5"):
        log("config 5: TurboQuant-4 decode B=8 64/8 d=128 ctx 131072")
        caches, q5, ms, nbytes = decode_case(cq, dev, stream, cq.TURBO4, 8, 64, 8, 128, 131072,
                                             steps_x, warm_x, chunk=8192)
        other["c5_turbo4"] = decode_summary(
            "BASELINE config 5: TurboQuant-4 KV decode", ms, nbytes,
            {"batch": 8, "q_heads": 64, "kv_heads": 8, "head_dim": 128, "context": 131072,
             "dtype": "4-bit codebook codes with f32 norms; f16 MFMA operands: codebook values "
                      "(f16-rounded f32 centroids), the rotated queries as one f16 operand and P "
                      "times the norms as one f16 operand (11 significant bits each); f32 "
                      "accumulate",
             "timed": "whole call (split-K decode + combine with unrotation)"})
        log(f"config 5: {ms * 1e3:.2f} us/call")
        if not args.no_cpu:
            sec, reps = cpu_baseline_decode(cq, caches[0], q5, cq.TURBO4, range(1), 131072,
                                            1.0 / 128 ** 0.5, threads)
            sec *= 8
            other["c5_turbo4"]["cpu_baseline"] = cpu_baseline_entry(
                round(nbytes / sec / 1e12, 6), "TB/s", sec * 1e6, threads, info,
                "oracle cache_attention (with the Hadamard unrotation of both sides) on 1 of the 8 "
                "sequences, scaled x8", reps)
            log(f"config 5 cpu: {sec * 1e6:.0f} us/call")
        del caches
        torch.cuda.empty_cache()

    if want("tp"):
        log("TurboProd keys + TurboQuant-4 values decode B=8 64/8 d=128 ctx 131072")
        caches, qp, ms, nbytes = decode_case(cq, dev, stream, cq.TURBOPROD, 8, 64, 8, 128,
                                             131072, steps_x, warm_x, chunk=8192,
                                             vfmt=cq.TURBO4)
        other["c5_shape_turboprod"] = decode_summary(
            "TurboProd (QJL) keys + TurboQuant-4 values decode at the BASELINE config-5 shape",
            ms, nbytes,
            {"batch": 8, "q_heads": 64, "kv_heads": 8, "head_dim": 128, "context": 131072,
             "dtype": "keys: 3-bit codebook codes, f32 norm and |r|, QJL sign bits as exact +-1 "
                      "operands; f16 MFMA operands: codebook values, rotated queries and S q as "
                      "one f16 operand each; values as TurboQuant-4; f32 accumulate",
             "timed": "whole call (split-K decode + combine with unrotation)"})
        log(f"turboprod: {ms * 1e3:.2f} us/call")
        if not args.no_cpu:
            sec, reps = cpu_baseline_decode(cq, caches[0], qp, cq.TURBOPROD, range(1), 131072,
                                            1.0 / 128 ** 0.5, threads, vfmt=cq.TURBO4)
            sec *= 8
            other["c5_shape_turboprod"]["cpu_baseline"] = cpu_baseline_entry(
                round(nbytes / sec / 1e12, 6), "TB/s", sec * 1e6, threads, info,
                "oracle cache_attention (QJL key scores, Hadamard unrotation) on 1 of the 8 "
                "sequences, scaled x8", reps)
            log(f"turboprod cpu: {sec * 1e6:.0f} us/call")
        del caches
        torch.cuda.empty_cache()

    if want("f8"):
        # flash_attn_with_config on E4M3 K / V with descales at the config-4 shape
        log("FP8 K/V attention at the config-4 shape")
        other["c4_shape_fp8_kv"] = fp8_attn_case(cq, dev, stream, max(steps_x, 20), max(warm_x, 40))
        log(f"fp8 kv: {other['c4_shape_fp8_kv']['us_per_call']} us/call")
        torch.cuda.empty_cache()
    if want("fx"):
        # the block-scaled formats of the reference beyond the BASELINE configs, at the config-2
        # decode shape
        for fmt, name in ((cq.MXFP8, "mxfp8"), (cq.NVFP4, "nvfp4")):
            log(f"{name} decode B=32 32/8 d=128 ctx 8192")
            caches, _, ms, nbytes = decode_case(cq, dev, stream, fmt, 32, 32, 8, 128, 8192,
                                                steps_x, warm_x)
            del caches
            dt = ("e4m3 codes with e8m0 block scales, exact in bf16; bf16 queries; P as bf16 "
                  "hi + lo operands; f32 accumulate" if fmt == cq.MXFP8 else
                  "e2m1 codes times e4m3 block scales, exact in f16, on both sides; queries as "
                  "f16 (scaled by a power of two into range), the f32 token scales on the scores "
                  "and, for values, in one f16 P operand (11 significant bits); f32 accumulate")
            other[f"c2_shape_{name}"] = decode_summary(
                f"{name.upper()}-KV decode at the BASELINE config-2 shape", ms, nbytes,
                {"batch": 32, "q_heads": 32, "kv_heads": 8, "head_dim": 128, "context": 8192,
                 "dtype": dt, "timed": "whole call (split-K decode + combine)"})
            log(f"{name}: {ms * 1e3:.2f} us/call")
            torch.cuda.empty_cache()
    if want("pd"):
        for dt in (torch.bfloat16, torch.float16):
            name = str(dt)[6:]
            log(f"plain {name} K/V decode B=32 32/8 d=128 ctx 8192")
            other[f"c2_shape_plain_{name}"] = plain_decode_case(cq, dev, stream, steps_x, warm_x,
                                                                dt)
            log(f"plain {name}: {other[f'c2_shape_plain_{name}']['us_per_call']} us/call")
    if want("pp"):
        for dt, d in ((torch.float16, 128), (torch.bfloat16, 64), (torch.bfloat16, 256)):
            name = f"{str(dt)[6:]}_d{d}"
            log(f"plain prefill {name} B=4 S=4096 32/8")
            other[f"c4_shape_plain_{name}"] = plain_prefill_case(cq, dev, stream,
                                                                 max(steps_x // 4, 5),
                                                                 max(warm_x // 4, 3), dt, d)
            log(f"plain prefill {name}: {other[f'c4_shape_plain_{name}']['us_per_call']} us/call")
    if want("fq"):
        f32 = torch.float32
        for dt in (torch.bfloat16, f32):
            name = str(dt)[6:]
            log(f"f32 queries over {name} K/V decode B=32 32/8 d=128 ctx 8192")
            other[f"c2_shape_f32q_{name}"] = plain_decode_case(cq, dev, stream, steps_x, warm_x,
                                                               dt, q_dtype=f32)
            log(f"f32q {name}: {other[f'c2_shape_f32q_{name}']['us_per_call']} us/call")
        log("f32 queries over bf16 K/V causal prefill B=4 S=4096 32/8 d=128")
        other["c4_shape_f32q_bfloat16"] = plain_prefill_case(cq, dev, stream, 5, 2,
                                                             torch.bfloat16, 128, q_dtype=f32)
        log(f"f32q prefill: {other['c4_shape_f32q_bfloat16']['us_per_call']} us/call")
    if want("ap"):
        log("append: B=32 x 8 kv heads x 2048 tokens, D=128, every format, keys and values")
        other["append_c2_shape"] = append_case(cq, dev, stream, steps_x, warm_x)
        log("append: " + ", ".join(f"{k} {v['us_per_call']} us"
                                   for k, v in other["append_c2_shape"]["per_side"].items()))
    if want("ra"):
        log("fused RoPE + FP8 append: prefill shape (config 4) and one decode step (config 2)")
        other["ra_prefill_c4"] = rope_append_case(cq, dev, stream, cq.FP8, 4, 32, 8, 128, 4096,
                                                  4096, steps_x, warm_x)
        other["ra_decode_step_c2"] = rope_append_case(cq, dev, stream, cq.FP8, 32, 32, 8, 128,
                                                      1, 8192, steps_x, warm_x)
        log(f"rope append: {other['ra_prefill_c4']['us_per_call']} us (prefill), "
            f"{other['ra_decode_step_c2']['us_per_call']} us (decode step)")
        torch.cuda.empty_cache()

    if res is None:
        res = {"metric": "partial run", "value": None, "note": "headline workload not selected"}
    if other:
        res["other_configs"] = other
    print(json.dumps(res), flush=True)


if __name__ == "__main__":
    main()
