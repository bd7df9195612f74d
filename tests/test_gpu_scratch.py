"""Calls without a workspace: their scratch comes from torch's caching allocator. Captured and replayed
with eager work between the replays, on side streams and from threads with allocator traffic, and with
no memory left for the scratch, against the same call in a caller's workspace or the eager result."""
import threading

import pytest
import torch

from tests.helpers import kv_source
from tests.test_gpu_graphs import randn, replays_match

pytestmark = pytest.mark.gpu


def calls(cq, dev, what):
    """Two calls of one kind over different inputs, fn(out or None) -> out, neither with a workspace."""
    def pair(make):
        return make(0), make(10)

    def dense(dtype, b, sq, sk, hq, hkv, d):
        def make(i):
            q, k, v = (randn(i + j, s, dtype, dev) for j, s in
                       enumerate(((b, sq, hq, d), (b, sk, hkv, d), (b, sk, hkv, d))))
            return lambda out: cq.flash_attn(q, k, v, 0.09, True, out=out)
        return pair(make)

    def side_pair(i, fmt, b, hkv, n, d):
        c = cq.TurboKvCache(fmt, fmt, b, hkv, d, n, device=dev)
        c.append(kv_source(i + 1, (b, hkv, n, d)).to(dev), kv_source(i + 2, (b, hkv, n, d)).to(dev))
        return c.k, c.v

    if what == "split bf16":
        return dense(torch.bfloat16, 1, 64, 4000, 8, 2, 128)
    if what == "f32 path":
        return dense(torch.float32, 2, 257, 3001, 6, 2, 128)
    if what == "f32 rows":
        return dense(torch.float32, 2, 1, 3000, 8, 2, 128)

    def make(i):
        if what == "varlen f16":
            cu = torch.tensor([0, 90, 91, 400], dtype=torch.int32, device=dev)
            ck = torch.tensor([0, 900, 1000, 4000], dtype=torch.int32, device=dev)
            q, k, v = (randn(i + j, s, torch.float16, dev) for j, s in
                       enumerate(((400, 8, 64), (4000, 2, 64), (4000, 2, 64))))
            return lambda out: cq.flash_attn_varlen(q, k, v, cu, ck, 309, 3000, 0.125, True, out=out)
        if what == "fp8 codes":
            q, k, v = (randn(i + j, s, torch.bfloat16, dev) for j, s in
                       enumerate(((2, 64, 8, 128), (2, 900, 2, 128), (2, 900, 2, 128))))
            k8, v8 = (x.to(torch.float8_e4m3fn) for x in (k, v))
            return lambda out: cq.flash_attn_fp8_codes(q, k8, v8, 0.09, True, out=out)
        q = randn(i + 5, (2, 16, 1, 128), dev=dev)
        if what == "decode":
            k, v = side_pair(i, cq.TURBO4, 2, 4, 2000, 128)
            return lambda out: cq.decode_attention(q, k, v, 2000, 0.1, out=out)
        if what == "paged":
            blocks = [(*side_pair(i + 3 * j, cq.FP8, 2, 4, n, 128), n) for j, n in enumerate((700, 300, 90))]
            return lambda out: cq.decode_attention_paged(q, blocks, 0.1, out=out)
        blocks = [(randn(i + 7 * n, (2, 4, n, 128), dev=dev), randn(i + n, (2, 4, n, 128), dev=dev), n)
                  for n in (320, 150, 64)]
        return lambda out: cq.flash_attn_blocks(q, blocks, 0.1, out=out)
    return pair(make)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_no_memory_left_for_the_scratch(cq, dev, dtype):
    """A call that fits without its images or partials is served where torch cannot give the scratch."""
    b, sq, sk, hq, hkv, d = 2, 600, 9000, 8, 4, 128
    q, k, v = (randn(i, s, dtype, dev) for i, s in
               enumerate(((b, sq, hq, d), (b, sk, hkv, d), (b, sk, hkv, d))))
    out, want = torch.empty_like(q), cq.flash_attn(q, k, v, 0.09, True)
    assert cq.flash_attn_workspace_bytes(dtype, b, sq, sk, hq, hkv, d) > 30 << 20
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(dev).total_memory
    taken = []
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(dev) + 1) / total, dev)
        with pytest.raises(torch.OutOfMemoryError):  # what earlier work left free in its segments
            while True:
                taken.append(torch.empty(16 << 20, dtype=torch.uint8, device=dev))
        cq.flash_attn(q, k, v, 0.09, True, out=out)
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
        del taken
    assert torch.equal(out, want)


@pytest.mark.parametrize("what", ["split bf16", "varlen f16", "f32 path", "f32 rows", "fp8 codes", "decode",
                                  "paged", "blocks"])
def test_capture_without_a_workspace(cq, dev, what):
    call, other = calls(cq, dev, what)
    out = call(None)
    replays_match(dev, lambda: call(out), [out], lambda: (other(None), torch.empty(1 << 20, device=dev)))


@pytest.mark.parametrize("what", ["split bf16", "f32 path", "decode", "paged"])
def test_side_streams(cq, dev, what):
    """Two calls of different inputs in flight on two streams, each stream's scratch freed and taken
    again while the other's kernels run."""
    call, other = calls(cq, dev, what)
    want = call(None).clone(), other(None).clone()
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(dev) for _ in range(2)]
    outs = [[], []]
    for _ in range(6):
        for i, (s, fn) in enumerate(zip(streams, (call, other))):
            with torch.cuda.stream(s):
                outs[i].append(fn(None))
                torch.empty(1 << 20, device=dev).fill_(float("nan"))  # takes the freed block over
    torch.cuda.synchronize()
    for got, w in zip(outs, want):
        assert all(torch.equal(g, w) for g in got)


def test_threads(cq, dev):
    fns = [f for what in ("split bf16", "f32 path", "decode", "paged") for f in calls(cq, dev, what)]
    want = [f(None).clone() for f in fns]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream(dev)):
            for _ in range(5):
                if not torch.equal(fns[i](None), want[i]):
                    bad.append(i)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(fns))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
