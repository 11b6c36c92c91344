"""Workgroups of the row-block forward: 64 or 128 rows, one set of waves or two that share a walk, by the size of the call."""
import numpy as np
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip
from gpu_utils import assert_close
from gpu_utils import pattern_forward
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


# Up to 256 workgroups of 64 rows, with a sequence of 1024 keys and more (four sets) and without one (two)
@pytest.mark.parametrize("lens,H,Hk,D,chunk,topk", [
    ([63, 64, 128, 129, 192, 193, 256, 257, 320, 321, 385], 2, 1, 64, 64, 3), ([449, 513, 577], 4, 4, 48, 64, 9), ([4096], 4, 2, 64, 128, 6),
    ([900], 1, 1, 16, 256, 2), ([700, 1, 640, 330], 16, 8, 64, 64, 4), ([1024, 2048], 8, 8, 32, 128, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_row_block_workgroups_of_four_sets(lens, H, Hk, D, chunk, topk, dtype):
    test_row_block_workgroups(lens, H, Hk, D, chunk, topk, dtype)


# Four sets over 64 rows: walks of fewer steps than sets, of one more, of every remainder beside a long one; queries that are the last rows of longer
# sequences, with more than 32 and 64 turns per set (a set's entries are read 64 turns at a time, every 32); a last chunk cut short
@pytest.mark.parametrize("lens_q,lens_k,H,Hk,D,chunk,topk", [
    ([63, 64, 128, 129, 192, 193, 256, 257, 320, 321, 385, 1100], None, 2, 1, 64, 64, 9), ([449, 513, 1077], None, 4, 4, 48, 64, 9), ([2100], None, 1, 1, 16, 256, 4),
    ([100, 1, 64], [8300, 70, 1500], 2, 2, 64, 64, 40), ([130], [18000], 2, 1, 32, 128, 60), ([65, 300], [1025, 300], 8, 8, 64, 128, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [True, False])
def test_row_block_workgroups_of_four_sets_over_long_walks(lens_q, lens_k, H, Hk, D, chunk, topk, dtype, causal):
    lens_k = lens_k or lens_q
    g = torch.Generator(device="cuda").manual_seed(sum(lens_k) + D)
    mk = lambda n, h: torch.randn((n, h, D), generator=g, device="cuda").to(dtype)
    q, k, v = mk(sum(lens_q), H), mk(sum(lens_k), Hk), mk(sum(lens_k), Hk)
    cu_q, cu_k = ([0] + [int(x) for x in np.cumsum(lens)] for lens in (lens_q, lens_k))
    args = (*(torch.tensor(x, dtype=torch.int32, device="cuda") for x in (cu_q, cu_k)), max(lens_q), max(lens_k))
    out = flash_moba.flash_moba_varlen_func(q, k, v, *args, chunk, topk, causal=causal)
    assert hip.last_fwd_row_blocks()
    pattern = flash_moba.flash_topk_varlen_func(q, k, *args, topk, chunk, causal=causal)
    # (the bound of the other attention tests)
    assert_close("out", out, pattern_forward(q, k, v, cu_q, cu_k, *pattern, chunk, causal)[0], 2e-2, 1e-2)
