"""The column layout of the MFMA prefill: a workgroup takes (query, head of the group) pairs,
query-major, so the ends of its wavefronts (32 columns) and blocks (256 columns, 128 at D = 256)
fall inside a query's heads for groups that do not divide them, and wavefronts whose queries see
fewer keys end before the workgroup. Against the oracle's unfused attention, within the bf16
bar of every attention test."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.helpers import assert_close_bf16

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


def test_split_in_a_callers_workspace(cq, dev):
    """The queried workspace gives the allocating call's bits; one that holds V^T but not the
    partials still serves the call, unsplit, within the bar."""
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
