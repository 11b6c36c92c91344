"""Column forward over groups of more query heads than a workgroup takes: the bits of a call with a key head for every query head."""
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip

pytestmark = pytest.mark.gpu


# groups of 65 (13 heads at a time), of a prime number above 64 (one at a time), of 128 in two halves, of 64 at once
@pytest.mark.parametrize("grp", [65, 67, 128, 64])
@pytest.mark.parametrize("D,chunk", [(64, 64), (128, 128)])
def test_groups_beyond_a_workgroup(grp, D, chunk):
    L, Hk = 20 * chunk + 37, 2
    g = torch.Generator(device="cuda").manual_seed(grp + D)
    q = torch.randn((L, Hk * grp, D), generator=g, device="cuda").to(torch.bfloat16)
    k, v = (torch.randn((L, Hk, D), generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    cu = torch.tensor([0, L], dtype=torch.int32, device="cuda")
    call = lambda k, v: flash_moba.flash_moba_varlen_func(q, k, v, cu, cu, L, L, chunk, 2)
    want = call(*(x.repeat_interleave(grp, dim=1) for x in (k, v)))
    assert not hip.last_fwd_row_blocks()
    got = call(k, v)
    assert not hip.last_fwd_row_blocks()
    assert torch.equal(got, want)
