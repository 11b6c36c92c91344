"""Row-block forward whose tiles two waves share, half of the keys each: two sets of them over 64 rows, from sequences of 1024 keys on."""
import pytest
import torch

import test_gpu_row_forms as forms
from flash_moba import flash_moba_hip as hip
from test_gpu_few_rows import _fwd_args

pytestmark = pytest.mark.gpu


# Heads to 64: as many workgroups as four sets are too many for, and no more than half as many again; above, where two sets are taken.  Walks of one step and of odd and even numbers, a set without
# a step, a last tile whose second half has no key or one; queries that are the last rows of longer sequences, rows before the first key; chunks of one to four tiles; heads of a group
@pytest.mark.parametrize("lens_q,lens_k,H,Hk,D,chunk,topk", [
    ([1024, 2048], None, 8, 8, 64, 128, 4), ([1057, 1, 64, 129], None, 16, 4, 40, 64, 9), ([500, 600, 1000], [1500, 601, 4033], 8, 8, 64, 256, 5),
    ([1027, 65, 31, 0, 97], None, 2, 2, 128, 64, 9), ([1100], None, 4, 1, 112, 128, 5), ([300, 70], [1025, 90], 4, 4, 128, 64, 12), ([1200, 64], [1000, 2000], 2, 1, 104, 256, 3),
    ([1027, 65, 33], None, 2, 2, 96, 64, 9), ([130, 1], [3000, 1056], 4, 2, 80, 64, 30)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [True, False])
def test_tiles_shared_by_two_waves(lens_q, lens_k, H, Hk, D, chunk, topk, dtype, causal):
    f = _fwd_args(lens_q, lens_k or lens_q, H, Hk, D, chunk, topk, causal)
    assert hip.load_library().fmoba_attn_fwd_row_sets(f) == 2
    if not hip.load_library().fmoba_attn_fwd_uses_row_blocks(f):
        pytest.skip("by columns")
    forms.test_row_block_workgroups_of_four_sets_over_long_walks(lens_q, lens_k, H, Hk, D, chunk, topk, dtype, causal)
