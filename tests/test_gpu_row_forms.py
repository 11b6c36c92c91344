"""Workgroups of the row-block forward: 64 or 128 rows, one set of waves or two that share a walk, by the size of the call."""
import numpy as np
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip
from gpu_utils import assert_close
from test_gpu_item_order import _reference

pytestmark = pytest.mark.gpu

# Two sets over 64 rows: walks of one step, of odd and even numbers of steps (a set without a step among them), lengths at the edges
# of 64 rows, chunks of one, two and four key blocks, the last of them cut short.  One set over 64 rows: many short sequences of
# narrow heads.  One set over 128 rows: every width, more than one word of selection bits per row
SMALL = [1, 63, 64, 65, 0, 127, 129, 193]
DOCS = [1, 64, 65, 300] * 10


@pytest.mark.parametrize("lens,H,Hk,D,chunk,topk", [
    (SMALL, 2, 2, 64, 64, 2), (SMALL, 4, 1, 128, 64, 3), (SMALL, 2, 1, 40, 128, 2), ([385, 700], 2, 2, 96, 256, 2), ([2100], 2, 2, 64, 64, 12),
    (DOCS, 16, 16, 64, 64, 2), (DOCS, 16, 4, 32, 128, 2), ([2300], 32, 8, 64, 64, 12), ([2300], 16, 16, 128, 64, 12),
    ([2300], 16, 16, 80, 64, 12)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_row_block_workgroups(lens, H, Hk, D, chunk, topk, dtype):
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + D)
    mk = lambda h: torch.randn((sum(lens), h, D), generator=g, device="cuda").to(dtype)
    q, k, v = mk(H), mk(Hk), mk(Hk)
    cu = [0] + [int(x) for x in np.cumsum(lens)]
    cud = torch.tensor(cu, dtype=torch.int32, device="cuda")
    args = (cud, cud, max(lens), max(lens))
    out = flash_moba.flash_moba_varlen_func(q, k, v, *args, chunk, topk, causal=True)
    pattern = flash_moba.flash_topk_varlen_func(q, k, *args, topk, chunk, causal=True)
    want = _reference(q, k, v, torch.zeros_like(q), cu, *pattern, chunk)[0]
    # (the bound of the other attention tests)
    assert_close("out", out, want, 2e-2, 1e-2)


def test_row_blocks_repeat_to_the_last_bit():
    """Workgroups whose waves drift apart (two to a unit, thousands of them): nothing may land in a tile that a wave still reads."""
    lens, H, D, chunk, topk = [13632, 9600, 5376, 2752], 16, 128, 64, 32
    g = torch.Generator(device="cuda").manual_seed(0)
    q, k, v = (torch.randn((sum(lens), H, D), generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
    run = lambda: flash_moba.flash_moba_varlen_func(q, k, v, cu, cu, max(lens), max(lens), chunk, topk, causal=True)
    with torch.no_grad():
        first = run()
        assert hip.last_fwd_row_blocks()
        assert all(torch.equal(run(), first) for _ in range(200))


# Four sets over 64 rows (up to 256 workgroups): walks of fewer steps than sets, of one more, of every remainder, queries that are the last rows of
# longer sequences' worth of steps; two sets on the other side of the line
@pytest.mark.parametrize("lens,H,Hk,D,chunk,topk", [
    ([63, 64, 128, 129, 192, 193, 256, 257, 320, 321, 385], 2, 1, 64, 64, 3), ([449, 513, 577], 4, 4, 48, 64, 9), ([4096], 4, 2, 64, 128, 6),
    ([900], 1, 1, 16, 256, 2), ([700, 1, 640, 330], 16, 8, 64, 64, 4), ([1024, 2048], 8, 8, 32, 128, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_row_block_workgroups_of_four_sets(lens, H, Hk, D, chunk, topk, dtype):
    test_row_block_workgroups(lens, H, Hk, D, chunk, topk, dtype)
