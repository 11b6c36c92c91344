"""Row-block forward whose tiles two waves share, half of the keys each: output and log-sum-exp, causal and not, by the form that is asserted to run."""
import numpy as np
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip
from gpu_utils import assert_close, pattern_forward
from test_gpu_few_rows import _fwd_args

pytestmark = pytest.mark.gpu


# walks of one step and of odd and even numbers, a set without a step, a last tile whose second half has no key or one, rows that see keys of one half alone; queries that are the
# last rows of longer sequences, rows before the first key; chunks of one to four tiles; heads of a group
@pytest.mark.parametrize("lens_q,lens_k,H,Hk,D,chunk,topk", [
    ([1027, 65, 31, 0, 97], None, 2, 2, 128, 64, 9), ([1100], None, 4, 1, 112, 128, 5), ([300, 70], [1025, 90], 4, 4, 128, 64, 12), ([1200, 64], [1000, 2000], 2, 1, 104, 256, 3),
    ([1027, 65, 33], None, 2, 2, 96, 64, 9), ([130, 1], [3000, 1056], 4, 2, 80, 64, 30), ([40, 1024], None, 8, 8, 128, 64, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [True, False])
def test_output_and_log_sum_exp(lens_q, lens_k, H, Hk, D, chunk, topk, dtype, causal):
    lens_k = lens_k or lens_q
    assert hip.load_library().fmoba_attn_fwd_key_halves(_fwd_args(lens_q, lens_k, H, Hk, D, chunk, topk, causal)) == 1
    g = torch.Generator(device="cuda").manual_seed(sum(lens_k) + D)
    mk = lambda n, h: torch.randn((n, h, D), generator=g, device="cuda").to(dtype)
    q, k, v = mk(sum(lens_q), H), mk(sum(lens_k), Hk), mk(sum(lens_k), Hk)
    cu_q, cu_k = ([0] + [int(x) for x in np.cumsum(lens)] for lens in (lens_q, lens_k))
    cud = [torch.tensor(x, dtype=torch.int32, device="cuda") for x in (cu_q, cu_k)]
    pattern = flash_moba.flash_topk_varlen_func(q, k, *cud, max(lens_q), max(lens_k), topk, chunk, causal=causal)
    out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, *pattern, *cud, None, None, None, max(lens_q), max(lens_k), 0.0, D ** -0.5, False, causal, 0.0, False, 128, chunk, None, _fwd_mode=2)
    assert hip.last_fwd_row_blocks() == 1
    want, want_lse = pattern_forward(q, k, v, cu_q, cu_k, *pattern, chunk, causal)
    # (the bounds of the other attention tests)
    assert_close("out", out, want, 2e-2, 1e-2)
    seen = torch.isfinite(want_lse)
    assert torch.equal(torch.isfinite(lse), seen) and (lse[~seen] == float("inf")).all()
    assert_close("lse", lse[seen], want_lse[seen], 2e-3, 1e-3)


# heads up to 64: more workgroups than units and no more than the longest walk covers
@pytest.mark.parametrize("lens,H,Hk,D,chunk,topk", [([1024, 2048], 8, 8, 64, 128, 4), ([1057, 1, 64], 16, 4, 40, 64, 9), ([2301], 8, 1, 32, 256, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_narrow_heads(lens, H, Hk, D, chunk, topk, dtype):
    test_output_and_log_sum_exp(lens, None, H, Hk, D, chunk, topk, dtype, True)
