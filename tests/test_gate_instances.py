"""The gate of up to 256 chunks, as built: taking the best scores off one by one costs no wave per SIMD against bisection, and is built where it can be reached."""
import re

from test_kernel_registers import _matching


def test_searches_of_the_cut():
    found = {}
    for k in _matching("topk_gate_kernelI"):
        m = re.search(r"topk_gate_kernelI(\w+?)Li(\d+)ELb([01])ELi(\d)EEEv", k[".name"])
        found[m.group(1), int(m.group(2)), int(m.group(4)), int(m.group(3))] = 512 // (-(-k[".vgpr_count"] // 8) * 8)
    assert {key[2:] for key in found} == {(2, 0), (2, 1), (4, 0), (4, 1), (8, 0)}  # (tiles of 32 chunks, one by one)
    for (dtype, dim, tiles, peel), waves in found.items():
        assert waves == found[dtype, dim, tiles, 0], (dtype, dim, tiles)
