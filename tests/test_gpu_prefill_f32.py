"""f32 queries on split bf16 operands (prefill_f32.hip): column and key remainders, the split of key
ranges, both workgroup widths, masks, score terms, head dims below the padded ones, variable lengths
and every K / V type, against float64 within the reference's f32 bar of 1e-5 of max |ref|; infinities
and NaN, also in values of masked keys;
and the route of a call whose workspace or alignment does not serve the path. Calls whose estimate is
smaller on the f32 MFMA kernel (short key ranges, few columns) run there; the sizes marked so are
checked to take the path."""
import math

import pytest
import torch

from tests.helpers import gpu_kernels, library_allocates

pytestmark = pytest.mark.gpu


def randn(seed, shape, dtype=torch.float32):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


def attention_f64(q, k, v, scale, causal, wl=-1, softcap=0.0, alibi=None):
    b, sq, hq, d = q.shape
    sk, hkv = k.shape[1], k.shape[2]
    q, k, v = (x.double().transpose(1, 2) for x in (q, k, v))
    k, v = (x.repeat_interleave(hq // hkv, 1) for x in (k, v))
    s = q @ k.transpose(2, 3) * scale
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    dist = torch.arange(sq)[:, None] + (sk - sq) - torch.arange(sk)[None]
    if alibi is not None:
        s -= alibi.double()[None, :, None, None] * dist.abs()
    hide = (dist < 0) & causal
    if wl >= 0:
        hide |= dist > wl
    s = s.masked_fill(hide, -math.inf)
    return torch.nan_to_num(s.softmax(-1)).matmul(v).transpose(1, 2)


def check(cq, dev, b, sq, sk, hq, hkv, d, kvd=torch.float32, causal=True, wl=-1, softcap=0.0,
          alibi=None, scale=1.0, taken=None):
    q = randn(1, (b, sq, hq, d)) * scale
    k, v = randn(2, (b, sk, hkv, d), kvd), randn(3, (b, sk, hkv, d), kvd)
    got = cq.flash_attn(q.to(dev), k.to(dev), v.to(dev), 1 / math.sqrt(d), causal, window_left=wl,
                        softcap=softcap, alibi_slopes=None if alibi is None else alibi.to(dev))
    if taken is not None:
        names = gpu_kernels(lambda: cq.flash_attn(
            q.to(dev), k.to(dev), v.to(dev), 1 / math.sqrt(d), causal, window_left=wl,
            softcap=softcap, alibi_slopes=None if alibi is None else alibi.to(dev)))
        assert ("prefill_f32_kernel" in names) == taken, names
    want = attention_f64(q, k, v, 1 / math.sqrt(d), causal, wl, softcap, alibi)
    assert (got.cpu().double() - want).abs().max() <= 1e-5 * want.abs().max()


@pytest.mark.parametrize("d", [8, 64, 72, 128])
@pytest.mark.parametrize("hq,hkv", [(2, 2), (6, 2), (16, 1)])
@pytest.mark.parametrize("sq,sk", [(129, 129), (86, 97), (257, 300), (65, 1000)])
def test_column_and_key_remainders(cq, dev, d, hq, hkv, sq, sk):
    check(cq, dev, 1, sq, sk, hq, hkv, d)


@pytest.mark.parametrize("d", [8, 64, 72, 128])
@pytest.mark.parametrize("b,hq,hkv,sq,sk", [
    (2, 6, 2, 129, 2500), (2, 6, 2, 257, 3001), (2, 6, 2, 513, 1111), (1, 16, 1, 86, 3001),
    (1, 16, 1, 65, 4000), (1, 16, 1, 129, 1300), (8, 2, 2, 700, 705), (4, 2, 2, 1033, 1033),
    (2, 2, 2, 383, 4000), (8, 2, 2, 511, 4000)])
def test_remainders_on_the_path(cq, dev, d, b, hq, hkv, sq, sk):
    check(cq, dev, b, sq, sk, hq, hkv, d, taken=True)


@pytest.mark.parametrize("b,sq,sk,hq,hkv,d", [(1, 195, 196, 8, 8, 128), (2, 300, 300, 8, 8, 128),
                                              (1, 40, 700, 32, 8, 128), (1, 20, 2000, 32, 2, 128),
                                              (1, 300, 128, 16, 1, 64), (1, 4, 3000, 16, 4, 64)])
def test_short_calls_stay_on_the_f32_mfma(cq, dev, b, sq, sk, hq, hkv, d):
    check(cq, dev, b, sq, sk, hq, hkv, d, taken=False)


@pytest.mark.parametrize("kvd", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("b,sq,sk,hq,hkv,d,causal,wl", [
    (1, 40, 5000, 8, 2, 128, True, -1),     # one block, up to 16 pieces
    (1, 700, 2100, 4, 4, 64, True, -1),     # pieces by falling size
    (2, 400, 1500, 8, 2, 128, True, 600),   # a window
    (1, 300, 200, 4, 2, 128, True, -1),     # queries that see no key
    (1, 200, 1111, 4, 2, 64, False, -1),
    (8, 600, 600, 16, 16, 64, True, -1),    # more than two blocks per CU: 8 wavefronts, unsplit
])
def test_splits_and_masks(cq, dev, kvd, b, sq, sk, hq, hkv, d, causal, wl):
    check(cq, dev, b, sq, sk, hq, hkv, d, kvd, causal, wl)


def test_score_terms_and_large_scores(cq, dev):
    slopes = 0.05 * (1 + torch.arange(6, dtype=torch.float32))
    check(cq, dev, 1, 150, 400, 6, 2, 64, softcap=3.0, alibi=slopes)
    check(cq, dev, 1, 150, 400, 6, 2, 128, scale=20.0)
    check(cq, dev, 2, 150, 2400, 6, 2, 64, softcap=3.0, alibi=slopes, taken=True)
    check(cq, dev, 2, 150, 2400, 6, 2, 128, scale=20.0, taken=True)


@pytest.mark.parametrize("lens", [[200, 0, 1, 333, 64], [700, 0, 1, 1333, 640, 90]])
def test_variable_lengths_equal_f64(cq, dev, lens):
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0)], dtype=torch.int32, device=dev)
    n, hq, hkv, d = sum(lens), 8, 2, 64
    q, k, v = randn(1, (n, hq, d)), randn(2, (n, hkv, d)), randn(3, (n, hkv, d))
    got = cq.flash_attn_varlen(q.to(dev), k.to(dev), v.to(dev), cu, cu, max(lens), max(lens), 0.125,
                               True).cpu()
    if max(lens) > 1000:
        assert "prefill_f32_kernel" in gpu_kernels(lambda: cq.flash_attn_varlen(
            q.to(dev), k.to(dev), v.to(dev), cu, cu, max(lens), max(lens), 0.125, True))
    at = 0
    for m in lens:
        if m:
            want = attention_f64(q[None, at:at + m], k[None, at:at + m], v[None, at:at + m], 0.125, True)
            assert (got[at:at + m].double() - want[0]).abs().max() <= 1e-5 * want.abs().max()
        at += m


@pytest.mark.parametrize("sq,sk", [(130, 200), (700, 2000)])
def test_non_finite_inputs(cq, dev, sq, sk):
    """A key at -inf * sign(q) gives probability 0, an infinite value an infinite output; queries near
    the top of f32 keep their scores (no part overflows: their bf16 rounding would)."""
    q = randn(1, (1, sq, 2, 64)).abs() + 0.5
    k, v = randn(2, (1, sk, 2, 64)), randn(3, (1, sk, 2, 64))
    k[0, 5] = -math.inf
    v[0, 9, 0, 3] = math.inf
    q[0, 100, 1, 5], k[0, :, 1, 5] = 3.4e38, k[0, :, 1, 5] * 2.0 ** -100
    got = cq.flash_attn(q.to(dev), k.to(dev), v.to(dev), 0.1, False).cpu()
    if sq > 130:
        assert "prefill_f32_kernel" in gpu_kernels(
            lambda: cq.flash_attn(q.to(dev), k.to(dev), v.to(dev), 0.1, False))
    keep = torch.arange(sk) != 5
    want = attention_f64(q, k[:, keep], v[:, keep], 0.1, False)
    assert torch.isposinf(got[0, :, 0, 3]).all()
    fin = torch.isfinite(want)
    assert (got.double() - want)[fin].abs().max() <= 1e-5 * want[fin].abs().max()


def test_workspaces_and_unaligned_rows(cq, dev):
    q, k, v = (randn(i, s).to(dev) for i, s in
               enumerate(((1, 200, 4, 64), (1, 900, 2, 64), (1, 900, 2, 64))))
    want = cq.flash_attn(q, k, v, 0.125, True)
    n = cq.flash_attn_workspace_bytes(torch.float32, 1, 200, 900, 4, 2, 64)
    ws = torch.empty(n, dtype=torch.uint8, device=dev)
    assert torch.equal(cq.flash_attn(q, k, v, 0.125, True, workspace=ws), want)
    images = 2 * 29 * 6 * 2 * 32 * 64
    assert n > images
    odd = torch.empty(1, 200, 4, 66, device=dev)[..., :64]
    odd.copy_(q)
    for got in (cq.flash_attn(q, k, v, 0.125, True, workspace=ws[:images]),
                cq.flash_attn(odd, k, v, 0.125, True)):
        assert (got - want).abs().max() <= 1e-5 * want.abs().max()


def test_workspaces_on_the_path(cq, dev, monkeypatch):
    """A call that takes the path in the queried workspace, in the images alone (unsplit) and in the
    library's own allocation."""
    b, sq, sk, hq, hkv, d = 2, 257, 3001, 6, 2, 128
    q, k, v = (randn(i, s).to(dev) for i, s in
               enumerate(((b, sq, hq, d), (b, sk, hkv, d), (b, sk, hkv, d))))
    call = lambda ws=None: cq.flash_attn(q, k, v, 0.125, True, workspace=ws)
    want = call()
    ws = torch.empty(cq.flash_attn_workspace_bytes(torch.float32, b, sq, sk, hq, hkv, d),
                     dtype=torch.uint8, device=dev)
    images = b * hkv * 94 * 6 * 2 * 32 * d
    assert torch.equal(call(ws), want)
    got = call(ws[:images])
    assert (got - want).abs().max() <= 1e-5 * want.abs().max()
    names = gpu_kernels(lambda: call(ws[:images]))
    assert "prefill_f32_kernel" in names and "prefill_f32_combine_kernel" not in names
    library_allocates(cq, monkeypatch)
    assert torch.equal(call(), want)
    assert "prefill_f32_combine_kernel" in gpu_kernels(call)


@pytest.mark.parametrize("kvd", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,sq,sk,hq,hkv,d,wl", [
    (2, 700, 2000, 6, 2, 64, -1), (2, 257, 3001, 6, 2, 128, -1), (2, 600, 2500, 6, 2, 72, 500),
    (1, 86, 3001, 16, 1, 128, -1), (8, 700, 705, 2, 2, 64, -1)])
def test_bad_value_of_a_masked_key(cq, dev, kvd, b, sq, sk, hq, hkv, d, wl):
    """Infinite and NaN values of keys that only some rows see: the other rows, some of them in the same
    tile, have the bits of the call with zeros there; rows that see them show them in that head dim."""
    q, k, v = (randn(i, s, t).to(dev) for i, s, t in
               ((1, (b, sq, hq, d), torch.float32), (2, (b, sk, hkv, d), kvd), (3, (b, sk, hkv, d), kvd)))
    bad = {sk - sq // 2: math.inf, sk - sq // 2 + 5: math.nan, sk - 1: -math.inf, sk - sq - 3: math.inf}
    pos = torch.arange(sq) + sk - sq
    clean = v.clone()
    seen = {}
    for i, (key, x) in enumerate(bad.items()):
        v[0, key, 0, 7 * i], clean[0, key, 0, 7 * i] = x, 0.0
        seen[7 * i] = (pos >= key) & ((pos - key <= wl) | (wl < 0))
    call = lambda v: cq.flash_attn(q, k, v, 0.1, True, window_left=wl)
    got, want = call(v).cpu(), call(clean).cpu()
    assert "prefill_f32_kernel" in gpu_kernels(lambda: call(v))
    for (key, x), (dim, s) in zip(bad.items(), seen.items()):
        hit = got[0, s][:, :hq // hkv, dim]
        assert hit.numel() and (hit.isnan() if math.isnan(x) else hit == x).all(), key
        got[0, s, :hq // hkv, dim] = want[0, s, :hq // hkv, dim] = 0.0
    assert torch.equal(got, want)


def test_bad_value_of_a_masked_key_elsewhere(cq, dev):
    """The same in E4M3 codes (NaN), in the last batch and head, and in a variable-length batch whose
    sequences start at other rows, with score terms."""
    b, sq, sk, hq, hkv, d = 2, 257, 3001, 6, 2, 128
    q, k, v = (randn(i, s).to(dev) for i, s in
               enumerate(((b, sq, hq, d), (b, sk, hkv, d), (b, sk, hkv, d))))
    k8, v8 = (x.to(torch.float8_e4m3fn).view(torch.uint8) for x in (k, v))
    v8[1, sk - 100, 1, 77] = 0
    want = cq.flash_attn_fp8_codes(q, k8, v8, 0.1, True, 0.5, 2.0).cpu()
    v8[1, sk - 100, 1, 77] = 0x7f
    call = lambda: cq.flash_attn_fp8_codes(q, k8, v8, 0.1, True, 0.5, 2.0)
    got = call().cpu()
    assert "prefill_f32_kernel" in gpu_kernels(call)
    assert got[1, sq - 100:, 3:, 77].isnan().all()
    got[1, sq - 100:, 3:, 77] = want[1, sq - 100:, 3:, 77] = 0.0
    assert torch.equal(got, want)

    lens = [700, 1, 1333, 640]
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0)], dtype=torch.int32, device=dev)
    n, d = sum(lens), 64
    q, k, v = (randn(i, (n, h, d)).to(dev) for i, h in ((1, 8), (2, 2), (3, 2)))
    slopes = (0.01 * torch.arange(1, 9, dtype=torch.float32)).to(dev)
    call = lambda: cq.flash_attn_varlen(q, k, v, cu, cu, 1333, 1333, 0.125, True, softcap=20.0,
                                        alibi_slopes=slopes)
    at = 701 + 900
    v[at, 1, 63] = 0.0
    want = call().cpu()
    v[at, 1, 63] = -math.inf
    got = call().cpu()
    assert "prefill_f32_kernel" in gpu_kernels(call)
    hit = slice(at, 701 + 1333)
    assert got[hit, 4:, 63].isneginf().all()
    got[hit, 4:, 63] = want[hit, 4:, 63] = 0.0
    assert torch.equal(got, want)
