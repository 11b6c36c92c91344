"""Which calls of the row-block forward have their tiles shared by two waves, at the lines of the rule."""
import ctypes

import pytest

from flash_moba import flash_moba_hip as H
from test_form_rules import fwd_args


# two sets over 64 rows above head dimension 64, from sequences of 1024 keys on; not narrower heads, whose compute units have room for two workgroups of four waves; not one set
@pytest.mark.parametrize("lens,heads,D,shared", [([1024], 8, 128, 1), ([1023], 8, 128, 0), ([1024, 1], 8, 72, 1), ([1024] * 3, 8, 96, 1), ([512] * 4, 8, 128, 0), ([4480], 8, 128, 1),
                                                 ([4736], 8, 128, 0), ([1024, 2048], 8, 64, 0), ([1100], 16, 64, 0), ([1536] * 2, 8, 64, 0), ([1024] * 3, 8, 32, 0), ([2048], 8, 64, 0)])
@pytest.mark.parametrize("causal", [0, 1])
def test_shared_tiles(lens, heads, D, shared, causal):
    f = fwd_args(lens, 64, 16, heads=heads, D=D, causal=causal)
    assert H.load_library().fmoba_attn_fwd_key_halves(ctypes.byref(f)) == shared
