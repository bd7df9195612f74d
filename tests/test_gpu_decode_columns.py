"""The decode's query staging and split combine at their edges: groups around the limits of the
column division (1, odd, 256 and above), column blocks that are not full, head dims below the
plane row, every query dtype, and split counts around the combine's 64 lanes and 8 rows in
flight. Against float64 attention over the cache's own dequantized rows, within the bf16 bar."""
import numpy as np
import pytest
import torch

from tests.helpers import assert_close_bf16

pytestmark = pytest.mark.gpu


def check(cq, dev, fmt, hq, hkv, d, lq, lk, splits=0, dtype=torch.bfloat16, alibi=None):
    g = torch.Generator().manual_seed(lk + hq)
    kv = [torch.randn(1, hkv, lk, d, generator=g).to(torch.bfloat16).to(dev) for _ in range(2)]
    cache = cq.TurboKvCache(fmt, fmt, 1, hkv, d, lk, device=dev)
    cache.append(*kv)
    q = torch.randn(1, hq, lq, d, generator=g).to(dtype)
    slopes = None if alibi is None else torch.linspace(0.01, alibi, hq)
    got = cache.attention(q.to(dev), 1.0 / d ** 0.5, window_right=0, splits=splits,
                          alibi_slopes=None if slopes is None else slopes.to(dev))
    k, v = (x.double().cpu().repeat_interleave(hq // hkv, 1) for x in cache.keys_values())
    s = q.double() @ k.transpose(2, 3) / d ** 0.5
    dist = torch.arange(lq)[:, None] + (lk - lq) - torch.arange(lk)[None]
    if slopes is not None:
        s -= slopes.double()[None, :, None, None] * dist.abs()
    s = s.masked_fill(dist < 0, -np.inf)
    want = s.softmax(-1) @ v
    assert_close_bf16(got.float().cpu().numpy(), want.numpy())


@pytest.mark.parametrize("hq,hkv,lq", [(2, 2, 1), (6, 2, 3), (5, 1, 7), (17, 1, 2), (256, 1, 2),
                                       (257, 1, 1), (300, 1, 2)])
@pytest.mark.parametrize("fmt,d", [(5, 128), (2, 64), (0, 256), (5, 80)])
def test_groups(cq, dev, fmt, d, hq, hkv, lq):
    check(cq, dev, fmt, hq, hkv, d, lq, 97, alibi=0.3 if hq == 6 else None)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("fmt", [5, 4, 3, 0])
def test_query_dtypes(cq, dev, fmt, dtype):
    check(cq, dev, fmt, 8, 2, 128, 1, 200, dtype=dtype)


@pytest.mark.parametrize("splits", [2, 7, 8, 9, 63, 64, 65, 130])
@pytest.mark.parametrize("fmt,d", [(5, 64), (0, 128), (2, 256)])
def test_combine_split_counts(cq, dev, fmt, d, splits):
    check(cq, dev, fmt, 4, 2, d, 1, 130 * 32, splits=splits)
