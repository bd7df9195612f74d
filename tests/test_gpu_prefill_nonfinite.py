"""Non-finite inputs of split prefill calls (long key ranges in pieces, merged at the end): a NaN key, a
key whose score is +inf, a NaN query row and infinite values give NaN and infinities where plain
attention does, whichever pieces they fall into, as the same call does unsplit (in a workspace that does
not hold the partials)."""
import math

import pytest
import torch

from tests.helpers import gpu_kernels

pytestmark = pytest.mark.gpu

SQ, SK, HQ, HKV, D = 70, 3000, 8, 2, 128
# V^T of the 16-bit kernel; the f32 kernel's images of 32-key tiles, three parts each, and a word per tile
UNSPLIT_BYTES = {
    torch.bfloat16: HKV * D * 3008 * 2, torch.float16: HKV * D * 3008 * 2,
    torch.float32: HKV * 94 * 6 * 2 * 32 * D + 768}
DTYPES = [torch.bfloat16, torch.float16, torch.float32]


def inputs(dtype):
    g = torch.Generator().manual_seed(5)
    q = torch.rand(1, SQ, HQ, D, generator=g) + 0.5  # positive: a key of +inf scores +inf
    k, v = (torch.randn(1, SK, HKV, D, generator=g) for _ in range(2))
    return q.to(dtype), k.to(dtype), v.to(dtype)


def both(cq, dev, q, k, v, causal=True):
    q, k, v = q.to(dev), k.to(dev), v.to(dev)
    n = cq.flash_attn_workspace_bytes(q.dtype, 1, SQ, SK, HQ, HKV, D)
    few = UNSPLIT_BYTES[q.dtype]
    assert n > few  # the plan splits this call
    ws = torch.empty(n, dtype=torch.uint8, device=dev)
    split = cq.flash_attn(q, k, v, 0.09, causal, workspace=ws).float().cpu()
    whole = cq.flash_attn(q, k, v, 0.09, causal, workspace=ws[:few]).float().cpu()
    return split, whole


@pytest.mark.parametrize("dtype", DTYPES)
def test_the_call_splits(cq, dev, dtype):
    q, k, v = (x.to(dev) for x in inputs(dtype))
    names = gpu_kernels(lambda: cq.flash_attn(q, k, v, 0.09, True))
    assert ("prefill_f32_combine_kernel" if dtype == torch.float32 else "prefill_combine_kernel") in names


def assert_same_kind(got, want, dtype):
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isposinf(), want.isposinf()) and torch.equal(got.isneginf(), want.isneginf())
    fin = want.isfinite()
    bar = {torch.bfloat16: 2e-2, torch.float16: 2e-3, torch.float32: 1e-5}[dtype]
    assert ((got - want)[fin].abs() <= bar * want[fin].abs().max()).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("at", [3, 1500, 2999])
@pytest.mark.parametrize("bad", [math.nan, math.inf])
def test_bad_key(cq, dev, dtype, at, bad):
    q, k, v = inputs(dtype)
    k[0, at, 1] = bad
    got, want = both(cq, dev, q, k, v)
    sees = torch.arange(SQ) + SK - SQ >= at
    assert got[0, sees][:, HQ // HKV:].isnan().all()  # NaN score, or inf - inf in the softmax
    assert got[0, :, :HQ // HKV].isfinite().all()     # the other kv head
    assert_same_kind(got, want, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_nan_query_row(cq, dev, dtype):
    q, k, v = inputs(dtype)
    q[0, 7, 2, 5] = math.nan
    got, want = both(cq, dev, q, k, v)
    assert got[0, 7, 2].isnan().all()
    assert got.isnan().sum() == D
    assert_same_kind(got, want, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("bad", [math.nan, math.inf, -math.inf])
def test_bad_value(cq, dev, dtype, bad):
    """Every query sees the key: its head dim becomes the value's kind in all rows of the kv head."""
    q, k, v = inputs(dtype)
    v[0, 700, 0, 9] = bad
    got, want = both(cq, dev, q, k, v, causal=False)
    hit = got[0, :, :HQ // HKV, 9]
    assert (hit.isnan() if math.isnan(bad) else hit == bad).all()
    assert got.isfinite().sum() == got.numel() - hit.numel()
    assert_same_kind(got, want, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_bad_value_of_vanishing_weight(cq, dev, dtype):
    """An infinite value in a piece whose weight underflows against another's: 0 times infinity, NaN as
    in the unsplit softmax."""
    q, k, v = inputs(dtype)
    k[0, 2500, 0] = 60.0   # one key far above the others
    v[0, 100, 0, 9] = math.inf
    got, want = both(cq, dev, q, k, v, causal=False)
    assert want[0, :, :HQ // HKV, 9].isnan().all()
    assert_same_kind(got, want, dtype)
