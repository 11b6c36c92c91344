"""Column lists made in one launch against those of scan and fill: the same lists, offsets and counts."""
import numpy as np
import pytest
import torch

from flash_moba import flash_moba_hip as hip
from flash_moba.mean_pool import flash_topk_mean_pool

pytestmark = pytest.mark.gpu


# Rows at the edges of a wave's 64 and a segment's 256, no rows, segments past the 32 that a workgroup counts at a time; chunks of one word and more, 64 columns of
# counts at a time and more than 128, sixteen words; prompts whose queries are the last rows of longer keys; slots that no list uses
@pytest.mark.parametrize("lens_q,lens_k,chunk,topk", [
    ([1], [1], 64, 1), ([63, 0, 65, 256], [63, 5, 65, 256], 64, 3), ([257, 255], [257, 255], 8, 4), ([700], [700], 10, 64), ([300, 77], [6400, 9000], 64, 9),
    ([500], [512 * 16], 16, 20), ([8500], [8500], 128, 8), ([10000], [10000], 400, 2)])
@pytest.mark.parametrize("causal", [True, False])
def test_lists_of_one_launch(lens_q, lens_k, chunk, topk, causal):
    H, D = 3, 64
    g = torch.Generator(device="cuda").manual_seed(sum(lens_k) + topk)
    q, k = (torch.randn((sum(n), H, D), generator=g, device="cuda").to(torch.bfloat16) for n in (lens_q, lens_k))
    cq, ck = (torch.tensor([0] + list(np.cumsum(n)), dtype=torch.int32, device="cuda") for n in (lens_q, lens_k))
    km, ckm, cols = flash_topk_mean_pool(k, ck, max(lens_k), chunk)
    # (a bound on the rows that makes more counts than one launch takes; nine rows and more: the same gate)
    one, two = max(9, max(lens_q)), 256 * (4096 // cols + 1)
    assert -(-one // 256) * cols <= 4096 and cols <= 512
    a, b = (hip.moba_fused_topk(q, km, cq, ck, ckm, n, max(lens_k), topk, chunk, causal, return_raw=False) for n in (one, two))
    assert all(torch.equal(x, y) for x, y in zip(a[:3], b[:3]))
