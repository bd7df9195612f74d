"""Calls without a workspace, whose scratch comes from torch's caching allocator, with no memory left
for it."""
import pytest
import torch

from tests.test_gpu_graphs import randn

pytestmark = pytest.mark.gpu


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
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(dev) + 1) / total, dev)
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(64 << 20, dtype=torch.uint8, device=dev)
        cq.flash_attn(q, k, v, 0.09, True, out=out)
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
    assert torch.equal(out, want)
