"""What the compiler made of kernels whose speed hangs on it, from the metadata of the built code objects: waves per SIMD, scalars spilled to lanes of
vector registers.  A change elsewhere in a kernel can cost either without any result changing."""
import struct

import pytest

from flash_moba import flash_moba_hip as H

msgpack = pytest.importorskip("msgpack")


def _kernels():
    """name -> metadata of every kernel of the library (notes named AMDGPU, type 32, of the code objects in it)"""
    data, at, found = open(H.LIB_PATH, "rb").read(), 0, {}
    while (at := data.find(b"AMDGPU\0\0", at)) >= 0:
        name_size, size, kind = struct.unpack("<III", data[at - 12:at])
        at += 8
        if (name_size, kind) == (7, 32):
            found.update((k[".name"], k) for k in msgpack.unpackb(data[at:at + size])["amdhsa.kernels"])
    return found


def _matching(part):
    found = [k for name, k in _kernels().items() if part in name]
    assert found, part
    return found


@pytest.mark.parametrize("dtype", ["DF16b", "DF16_"])
@pytest.mark.parametrize("near", [0, 1])
def test_dkdv_of_narrow_heads_keeps_three_waves_per_simd(dtype, near):
    # 512 registers per SIMD lane, given out in eights: three waves of at most 168
    for k in _matching("attn_bwd_dkdv_kernelI%sLi64ELb0ELb0ELb%dE" % (dtype, near)):
        assert k[".vgpr_count"] <= 168 and k[".vgpr_spill_count"] == 0


@pytest.mark.parametrize("chunks", [64, 128, 256])
def test_gate_spills_nothing(chunks):
    for k in _matching("topk_gate_kernelI"):
        if "ELi%dEEEv" % (chunks // 32) in k[".name"]:
            assert (k[".sgpr_spill_count"], k[".vgpr_spill_count"], k[".private_segment_fixed_size"]) == (0, 0, 0), k[".name"]
