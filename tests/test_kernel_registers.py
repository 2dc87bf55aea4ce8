"""Registers of the tiled GEMM's kernels, read from the code objects of the built library: two workgroups of four waves have to
fit a compute unit, i.e. a wave may hold 256 of the 512 registers of its SIMD (accumulation registers included)."""
import struct

import msgpack
import pytest

from deep8_amd import capi

NT_AMDGPU_METADATA = 32


def _code_objects(blob):
    at = blob.find(b"\x7fELF", 1)
    while at >= 0:
        if blob[at + 4] == 2 and struct.unpack_from("<H", blob, at + 18)[0] == 224:  # 64-bit, EM_AMDGPU
            yield at
        at = blob.find(b"\x7fELF", at + 1)


def _kernels(blob, at):
    """the kernels' metadata of the code object that starts at `at`"""
    shoff, = struct.unpack_from("<Q", blob, at + 40)
    shentsize, shnum = struct.unpack_from("<HH", blob, at + 58)
    for i in range(shnum):
        kind, _, _, offset, size = struct.unpack_from("<IQQQQ", blob, at + shoff + i * shentsize + 4)
        p, end = at + offset, at + offset + size
        while kind == 7 and p < end:  # SHT_NOTE
            namesz, descsz, typ = struct.unpack_from("<III", blob, p)
            desc = p + 12 + (namesz + 3) // 4 * 4
            if typ == NT_AMDGPU_METADATA and blob[p + 12:p + 12 + namesz].rstrip(b"\0") == b"AMDGPU":
                yield from msgpack.unpackb(blob[desc:desc + descsz], raw=False, strict_map_key=False)["amdhsa.kernels"]
            p = desc + (descsz + 3) // 4 * 4


def test_two_workgroups_of_the_tiled_kernels_fit_a_compute_unit():
    with open(capi.LIB_PATH, "rb") as f:
        blob = f.read()
    found = {k[".name"]: k for at in _code_objects(blob) for k in _kernels(blob, at) if "gemm_tiled" in k[".name"]}
    if not found:
        pytest.skip("the library's code objects are compressed")
    assert any("gemm_tiled_pair_kernel" in n for n in found) and len(found) > 100
    over = {n: k[".vgpr_count"] for n, k in found.items() if k[".vgpr_count"] > 256 or k[".vgpr_spill_count"]}
    assert not over


def test_two_workgroups_on_images_of_few_channels_fit_a_compute_unit():
    """up to 64 KB of image rows a tile are asked for at the launch; the kernel's own arrays must leave them to two workgroups"""
    with open(capi.LIB_PATH, "rb") as f:
        blob = f.read()
    found = {k[".name"]: k for at in _code_objects(blob) for k in _kernels(blob, at) if "conv_direct_forward_kernel" in k[".name"]}
    if not found:
        pytest.skip("the library's code objects are compressed")
    assert not {n: k[".group_segment_fixed_size"] for n, k in found.items() if 2 * (k[".group_segment_fixed_size"] + 64 * 1024) > 160 * 1024}
    assert not {n: k[".vgpr_count"] for n, k in found.items() if k[".vgpr_count"] > 256 or k[".vgpr_spill_count"]}
