"""Registers and LDS of the built decode kernels, read from the code objects in libcqkv.so: the split
counts assume that a CU holds two 8-wavefront workgroups' worth of waves where the registers allow
it, so the kernels whose allocation lies just below a limit may not slip over it, nor spill."""
import os
import struct

import pytest

msgpack = pytest.importorskip("msgpack")

SO = os.path.join(os.path.dirname(__file__), "..", "candle-rocm-vulkan_amd", "libcqkv.so")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
CU_LDS, SIMD_VGPRS = 160 * 1024, 512


def code_objects(blob):
    """The gfx950 ELF images of the offload bundles in a library."""
    at = blob.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", blob, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, p)
            name = blob[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in name and size:
                yield blob[at + off:at + off + size]
        at = blob.find(MAGIC, at + 1)


def kernel_metadata(elf):
    """amdhsa.kernels of an ELF image's AMDGPU note (type 32, msgpack)."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        sh = shoff + i * shentsize
        kind, = struct.unpack_from("<I", elf, sh + 4)
        off, size = struct.unpack_from("<QQ", elf, sh + 24)
        if kind != 7:  # SHT_NOTE
            continue
        p = off
        while p < off + size:
            namesz, descsz, note = struct.unpack_from("<III", elf, p)
            desc = p + 12 + (namesz + 3) // 4 * 4
            if note == 32:
                yield from msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]
            p = desc + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def decode_kernels():
    if not os.path.exists(SO):
        pytest.skip("libcqkv.so is not built")
    with open(SO, "rb") as f:
        blob = f.read()
    found = {k[".name"]: k for elf in code_objects(blob) for k in kernel_metadata(elf)
             if "decode_kernelI" in k[".name"]}
    assert len(found) > 300
    return found


def workgroups_per_cu(k, waves):
    regs = (k[".vgpr_count"] + 7) // 8 * 8  # VGPRs and AGPRs together, allocated in eights
    return min(SIMD_VGPRS // regs * 4 // waves, CU_LDS // max(1, k[".group_segment_fixed_size"]))


TURBO4, MXFP4, NVFP4, MXFP8, TURBOC = 0, 2, 3, 4, 6


@pytest.mark.parametrize("kf,vf,d,waves,terms,want", [
    *[(k, v, 256, 4, t, 2) for k, v in ((TURBO4, TURBO4), (TURBO4, MXFP4), (TURBO4, TURBOC),
                                        (MXFP4, TURBO4), (MXFP4, MXFP4), (NVFP4, TURBO4),
                                        (NVFP4, MXFP4), (TURBOC, TURBO4)) for t in (0, 1)],
    (MXFP4, MXFP4, 128, 4, 0, 3), (MXFP4, MXFP8, 128, 4, 0, 3), (MXFP4, MXFP4, 64, 4, 0, 4),
    (MXFP8, MXFP8, 64, 8, 0, 2),
])
def test_decode_workgroups_per_cu(decode_kernels, kf, vf, d, waves, terms, want):
    tag = f"decode_kernelILi{kf}ELi{vf}ELi{d}ELi{waves}ELb{terms}ELb0EE"
    k, = [m for n, m in decode_kernels.items() if tag in n]
    assert workgroups_per_cu(k, waves) >= want
    assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0
