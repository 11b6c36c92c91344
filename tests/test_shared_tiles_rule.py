"""Which calls of the row-block forward have their tiles shared by two waves, at the lines of the rule."""
import ctypes

import pytest

from flash_moba import flash_moba_hip as H
from test_form_rules import fwd_args


# two sets over 64 rows above head dimension 64, from sequences of 1024 keys on; not one set
@pytest.mark.parametrize("lens,heads,D,shared", [([1024], 8, 128, 1), ([1023], 8, 128, 0), ([1024, 1], 8, 72, 1), ([1024] * 3, 8, 96, 1), ([512] * 4, 8, 128, 0), ([4480], 8, 128, 1),
                                                 ([4736], 8, 128, 0)])
@pytest.mark.parametrize("causal", [0, 1])
def test_shared_tiles(lens, heads, D, shared, causal):
    f = fwd_args(lens, 64, 16, heads=heads, D=D, causal=causal)
    assert H.load_library().fmoba_attn_fwd_key_halves(ctypes.byref(f)) == shared


# narrower heads, whose compute units have room for two workgroups of four waves: where the longest walk covers the workgroups that start later, which those of calls that are not causal
# never do, nor those of queries that are the last rows of longer sequences; items that start longest first
@pytest.mark.parametrize("lens,heads,shared", [([1024, 2048], 8, 1), ([2500, 500], 8, 1), ([3000], 8, 1), ([1100], 16, 1), ([1700, 900], 8, 1), ([1024, 1200], 8, 0), ([1112, 1512], 8, 0), ([1200] * 2, 8, 0), ([1536] * 2, 8, 0), ([1024] * 3, 8, 0),
                                               ([1400], 16, 0), ([1024], 24, 0), ([3200], 8, 1), ([3201], 8, 0), ([3000, 600], 8, 0), ([2600], 9, 0), ([2000, 1200], 8, 0), ([2641, 407, 1199, 790], 4, 0)])
@pytest.mark.parametrize("D", [32, 64])
def test_shared_tiles_of_narrow_heads(lens, heads, shared, D):
    f = fwd_args(lens, 64, 16, heads=heads, D=D)
    halves = H.load_library().fmoba_attn_fwd_key_halves
    assert halves(ctypes.byref(f)) == shared
    f.is_causal = 0
    assert halves(ctypes.byref(f)) == 0
    f.is_causal = 1
    f.total_k = f.max_seqlen_k = max(lens) + 64
    assert halves(ctypes.byref(f)) == 0
