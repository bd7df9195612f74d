"""The column layout of the MFMA prefill: a workgroup takes (query, head of the group) pairs,
query-major, so the ends of its wavefronts (32 columns) and blocks (256 columns, 128 at D = 256)
fall inside a query's heads for groups that do not divide them, and wavefronts whose queries see
fewer keys end before the workgroup. Against the oracle's unfused attention, within the bf16
bar of every attention test."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import assert_close_bf16, gpu_kernels, library_allocates

pytestmark = pytest.mark.gpu


def randn(seed, shape):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g).to(torch.bfloat16)


def check(cq, dev, b, sq, sk, hq, hkv, d, wl=-1, wr=0, alibi=None, dtype=torch.bfloat16):
    q, k, v = (randn(i, s).to(dtype) for i, s in
               enumerate(((b, sq, hq, d), (b, sk, hkv, d), (b, sk, hkv, d))))
    scale = 1.0 / d ** 0.5
    got = cq.flash_attn(q.to(dev), k.to(dev), v.to(dev), scale, wr == 0, window_left=wl,
                        window_right=wr,
                        alibi_slopes=None if alibi is None else torch.tensor(alibi).to(dev))
    qf, kf, vf = (x.float().permute(0, 2, 1, 3).contiguous().numpy() for x in (q, k, v))
    want = O.attention_unfused(qf, kf, vf, scale, wl=wl, wr=wr, threads=16,
                               **({} if alibi is None else
                                  {"alibi": np.array(alibi, np.float32)}))
    assert_close_bf16(got.float().cpu().numpy(), O.round_bf16(want).transpose(0, 2, 1, 3))


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("hq,hkv", [(2, 2), (6, 2), (5, 1), (16, 2), (40, 1)])
@pytest.mark.parametrize("sq", [17, 86, 257])
def test_groups_and_block_ends(cq, dev, d, hq, hkv, sq):
    check(cq, dev, 1, sq, sq + 70, hq, hkv, d)


@pytest.mark.parametrize("hq,hkv", [(2, 2), (6, 2), (16, 2)])
@pytest.mark.parametrize("sq,sk,wl,wr", [(300, 300, 40, 0), (260, 513, 100, 7), (300, 70, -1, 0),
                                         (90, 200, -1, -1), (520, 520, 3, 0)])
def test_wavefront_key_ranges(cq, dev, hq, hkv, sq, sk, wl, wr):
    check(cq, dev, 2, sq, sk, hq, hkv, 64, wl, wr)


@pytest.mark.parametrize("hq,hkv", [(4, 4), (6, 2), (16, 2)])
def test_alibi_slope_per_column(cq, dev, hq, hkv):
    check(cq, dev, 1, 130, 200, hq, hkv, 128,
          alibi=[2.0 ** -(1 + i % 8) for i in range(hq)], dtype=torch.float16)


@pytest.mark.parametrize("d,hq,hkv,sq,sk,wl,wr", [
    (128, 8, 2, 40, 5000, -1, 0),    # few column blocks, long ranges: up to 16 pieces
    (64, 2, 2, 300, 3001, -1, 0),    # several blocks, ragged last tile
    (256, 4, 1, 33, 2100, -1, -1),
    (128, 8, 8, 1100, 1100, -1, 0),  # causal: the early blocks have one piece, the late ones more
    (128, 8, 2, 64, 4100, 1500, 0),  # a window: the range begins inside the keys
    (128, 4, 1, 1000, 700, -1, 0),   # the first queries see no key
])
def test_split_key_ranges(cq, dev, d, hq, hkv, sq, sk, wl, wr):
    check(cq, dev, 1, sq, sk, hq, hkv, d, wl, wr)


def test_split_in_a_callers_workspace(cq, dev, monkeypatch):
    """The queried workspace gives the bits of the call that allocates for itself, in the library as
    from the front end; one that holds V^T but not the partials still serves the call, unsplit, within
    the bar."""
    q, k, v = (randn(i, s).to(dev) for i, s in
               enumerate(((1, 64, 8, 128), (1, 4000, 2, 128), (1, 4000, 2, 128))))
    want = cq.flash_attn(q, k, v, 0.09, True)
    n = cq.flash_attn_workspace_bytes(torch.bfloat16, 1, 64, 4000, 8, 2, 128)
    ws = torch.empty(n, dtype=torch.uint8, device=dev)
    assert torch.equal(cq.flash_attn(q, k, v, 0.09, True, workspace=ws), want)
    vt = 2 * 128 * 4032 * 2
    assert n > vt
    got = cq.flash_attn(q, k, v, 0.09, True, workspace=ws[:vt])
    assert_close_bf16(got.float().cpu().numpy(), want.float().cpu().numpy())
    library_allocates(cq, monkeypatch)
    assert torch.equal(cq.flash_attn(q, k, v, 0.09, True), want)
    assert "prefill_combine_kernel" in gpu_kernels(lambda: cq.flash_attn(q, k, v, 0.09, True))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_windowed_split_in_the_librarys_memory(cq, dev, dtype, monkeypatch):
    """A window's plan is not one that the workspace query sizes for (causal and full): the library's
    own allocation, sized by the call's plan, and the queried workspace both serve it."""
    q, k, v = (randn(i, s).to(dev).to(dtype) for i, s in
               enumerate(((2, 400, 8, 128), (2, 9000, 2, 128), (2, 9000, 2, 128))))
    call = lambda: cq.flash_attn(q, k, v, 0.09, True, window_left=3000)
    want = call()
    library_allocates(cq, monkeypatch)
    got = call()
    assert {"prefill_combine_kernel", "prefill_f32_combine_kernel"} & gpu_kernels(call)
    bar = 2e-2 if dtype == torch.bfloat16 else 1e-5
    assert (got - want).abs().max() <= bar * want.abs().max()


@pytest.mark.parametrize("d", [64, 128, 256])
def test_split_with_score_terms(cq, dev, d):
    check(cq, dev, 1, 40, 3000, 6, 2, d, alibi=[2.0 ** -(4 + i) for i in range(6)])


def test_split_variable_lengths(cq, dev):
    """Few queries against long key ranges of different lengths (more key tiles per block than the
    longest query and key lengths together suggest), an empty sequence and one without keys."""
    lens_q, lens_k, hq, hkv, d = [40, 0, 130, 70], [3000, 60, 700, 0], 8, 2, 128
    q, k, v = randn(1, (sum(lens_q), hq, d)), randn(2, (sum(lens_k), hkv, d)), randn(3, (sum(lens_k), hkv, d))
    cu = [torch.tensor([0, *np.cumsum(n)], dtype=torch.int32, device=dev) for n in (lens_q, lens_k)]
    got = cq.flash_attn_varlen(q.to(dev), k.to(dev), v.to(dev), *cu, max(lens_q), max(lens_k), 0.09,
                               True).float().cpu().numpy()
    iq = ik = 0
    for nq, nk in zip(lens_q, lens_k):
        if nq:
            qf, kf, vf = (x.float().permute(1, 0, 2)[None].contiguous().numpy() for x in
                          (q[iq:iq + nq], k[ik:ik + nk], v[ik:ik + nk]))
            want = (O.round_bf16(O.attention_unfused(qf, kf, vf, 0.09, wl=-1, wr=0, threads=16))[0]
                    .transpose(1, 0, 2) if nk else np.zeros((nq, hq, d), np.float32))
            assert_close_bf16(got[iq:iq + nq], want)
        iq, ik = iq + nq, ik + nk


def test_split_with_e4m3_keys_and_cache_append(cq, dev):
    """Split calls whose workspace also holds the widened E4M3 K, and whose pre-pass appends."""
    b, sq, sk, hq, hkv, d = 1, 40, 3000, 8, 2, 128
    q, k, v = randn(1, (b, sq, hq, d)), randn(2, (b, sk, hkv, d)), randn(3, (b, sk, hkv, d))
    k8, v8 = (x.to(dev).to(torch.float8_e4m3fn) for x in (k, v))
    got = cq.flash_attn_fp8_codes(q.to(dev), k8, v8, 0.09, True)
    want = cq.flash_attn(q.to(dev), k8.to(torch.bfloat16), v8.to(torch.bfloat16), 0.09, True)
    assert_close_bf16(got.float().cpu().numpy(), want.float().cpu().numpy())
    sides = [cq.CacheSide.empty(cq.FP8, bool(i & 1), b, hkv, d, sk, dev) for i in range(4)]
    plain = cq.flash_attn(q.to(dev), k.to(dev), v.to(dev), 0.09, True)
    fused = cq.flash_attn(q.to(dev), k.to(dev), v.to(dev), 0.09, True, k_cache=sides[0],
                          v_cache=sides[1])
    assert torch.equal(fused, plain)
    for side, x in ((sides[2], k), (sides[3], v)):
        cq.quant_append(side, x.to(dev).transpose(1, 2), 0)
    for a, r in zip(sides[:2], sides[2:]):
        assert torch.equal(a.codes, r.codes) and torch.equal(a.scales, r.scales)
