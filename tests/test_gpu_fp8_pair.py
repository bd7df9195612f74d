"""cqkv_fp8_quantize_pair: K and V of different sizes in one set of launches give the codes and
scales of the single-tensor calls, which match the oracle; sizes around the 8-element pieces, and
rows whose codes or elements are not aligned for them."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("nk,nv", [(1, 8), (7, 4096), (2049, 15), (100003, 70000), (0, 9)])
def test_pair_equals_oracle(cq, dev, dtype, nk, nv):
    g = torch.Generator().manual_seed(nk + nv)
    xs = [(torch.randn(n, generator=g) * 3).to(dtype) for n in (nk, nv)]
    xs[1][0] = -0.0
    if nk:
        got = cq._fp8_quantize_pair(*(x.to(dev) for x in xs))
        pairs = [(got[0], got[2]), (got[1], got[3])]
    else:  # an empty side is null data: the single calls
        pairs = [None, cq.fp8_quantize_tensor(xs[1].to(dev))]
    for x, p in zip(xs, pairs):
        if p is None:
            continue
        codes, scale = O.fp8_quantize_tensor(x.float().numpy())
        np.testing.assert_array_equal(p[0].cpu().numpy(), codes)
        assert p[1][0].item() == np.float32(scale)


@pytest.mark.parametrize("off", [1, 4])
def test_unaligned_elements(cq, dev, off):
    x = torch.randn(999 + off, generator=torch.Generator().manual_seed(3)).to(torch.bfloat16).to(dev)
    codes, scale = cq.fp8_quantize_tensor(x[off:])
    want, ws = O.fp8_quantize_tensor(x[off:].float().cpu().numpy())
    np.testing.assert_array_equal(codes.cpu().numpy(), want)
    assert scale[0].item() == np.float32(ws)
