"""Where the column lists enter the row blocks of the dQ pass, and the padded layout of softmax_d: both come from the delta pass."""
import numpy as np
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip
from gpu_utils import assert_close
from test_gpu_item_order import _reference

pytestmark = pytest.mark.gpu

MANY = [0, 1, 63, 64, 65, 255, 256, 257, 300, 513]


# rows at the edges of 256-row blocks; more sequences than one step of the search for a column's sequence takes (64 and 64 * 64 are its
# steps), empty ones among them; queries that are the last rows of longer sequences; more boundaries than a wave has lanes
@pytest.mark.parametrize("lens_q,lens_k,D,chunk,topk", [
    (MANY * 13, MANY * 13, 32, 64, 3), ([1] * 4200, [1] * 4200, 32, 64, 2), ([255, 0, 257], [900, 70, 257], 64, 128, 2),
    ([100, 513], [1100, 600], 96, 64, 4), ([17000], [17000], 32, 256, 8), ([300], [300], 128, 64, 3)])
def test_dq_over_row_blocks_agrees_with_partial_rows(lens_q, lens_k, D, chunk, topk):
    H = 2
    g = torch.Generator(device="cuda").manual_seed(sum(lens_q) + D)
    mk = lambda n: torch.randn((n, H, D), generator=g, device="cuda").to(torch.bfloat16)
    q, k, v, dout = mk(sum(lens_q)), mk(sum(lens_k)), mk(sum(lens_k)), mk(sum(lens_q))
    cq, ck = (torch.tensor([0] + list(np.cumsum(x)), dtype=torch.int32, device="cuda") for x in (lens_q, lens_k))
    mq, mkk, scale = max(lens_q), max(lens_k), D ** -0.5
    causal = mq > 1  # (as the attention entry points have it)
    csc = flash_moba.flash_topk_varlen_func(q, k, cq, ck, mq, mkk, topk, chunk, causal=causal)
    out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, *csc, cq, ck, None, None, None, mq, mkk, 0.0, scale, False, causal, 0.0, False, 128, chunk, None)
    run = lambda mode: hip.moba_varlen_bwd(dout, q, k, v, out, lse, None, None, None, *csc, cq, ck, None, mq, mkk, 0.0, scale, False, causal, 0.0, False,
                                           128, chunk, None, _dq_mode=mode)
    dq, dk, dv, sd = run(1)
    want = run(2)
    # (the bounds of the other attention tests: 16-bit results of sums of 16-bit factors, and 16-bit partial rows on one side)
    for name, x, y in zip(("dq", "dk", "dv"), (dq, dk, dv), want):
        assert_close(name, x, y, 2e-2, 1e-2)
    assert torch.equal(sd, want[3])
    delta = (out.float() * dout.float()).sum(-1).T
    layout, pad = torch.zeros_like(sd), torch.ones(sd.shape[1], dtype=torch.bool, device="cuda")
    for b, (s, n) in enumerate(zip(np.cumsum([0] + lens_q), lens_q)):
        layout[:, s + 128 * b:s + 128 * b + n] = delta[:, s:s + n]
        pad[s + 128 * b:s + 128 * b + n] = False
    # (fp32 sums of D products in another order: a few 2^-24 of the sum of their magnitudes, which is below D here)
    assert (sd - layout).abs().max() < 1e-5 * D
    assert (sd[:, pad] == 0).all()


# The places are looked up from the first row block that sees a column to the end of its sequence: one sequence far longer than the others,
# columns that begin inside a row block, queries that are the last rows (columns before the first row, after the last), and the plain rule
@pytest.mark.parametrize("lens_q,lens_k,chunk,topk", [([5000] + [70] * 9, [5000] + [70] * 9, 64, 4), ([700, 3], [1500, 2000], 64, 3), ([900], [400], 192, 2)])
@pytest.mark.parametrize("causal", [True, False])
def test_places_between_a_columns_first_row_and_the_end(lens_q, lens_k, chunk, topk, causal):
    H, D = 2, 64
    g = torch.Generator(device="cuda").manual_seed(sum(lens_q) + chunk)
    mk = lambda n: torch.randn((n, H, D), generator=g, device="cuda").to(torch.bfloat16)
    q, k, v, dout = mk(sum(lens_q)), mk(sum(lens_k)), mk(sum(lens_k)), mk(sum(lens_q))
    cq, ck = (torch.tensor([0] + list(np.cumsum(x)), dtype=torch.int32, device="cuda") for x in (lens_q, lens_k))
    mq, mkk, scale = max(lens_q), max(lens_k), D ** -0.5
    csc = flash_moba.flash_topk_varlen_func(q, k, cq, ck, mq, mkk, topk, chunk, causal=causal)
    out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, *csc, cq, ck, None, None, None, mq, mkk, 0.0, scale, False, causal, 0.0, False, 128, chunk, None)
    res = []
    for mode in (1, 2):
        held = [torch.full((1 << 17,), -1, dtype=torch.int32, device="cuda") for _ in range(64)]  # (what the workspace may hold before)
        del held
        res.append(hip.moba_varlen_bwd(dout, q, k, v, out, lse, None, None, None, *csc, cq, ck, None, mq, mkk, 0.0, scale, False, causal, 0.0, False,
                                       128, chunk, None, _dq_mode=mode))
    for name, x, y in zip(("dq", "dk", "dv"), *res):  # (bounds as above)
        assert_close(name, x, y, 2e-2, 1e-2)


# Walks of the dQ pass around 32 and 64 steps and past 64 (its records come 64 at a time, every 32 steps), of several batches of columns
# (256 of them, 512 steps), with rows that are in few of the steps or, past the first 64, in none
@pytest.mark.parametrize("L,chunk,topk", [(31 * 64, 64, 3), (32 * 64 + 1, 64, 3), (64 * 64, 64, 2), (65 * 64 + 7, 128, 1), (4200, 192, 2), (16700, 64, 2)])
@pytest.mark.parametrize("D", [64, 96, 128, 256])
def test_dq_over_long_walks(L, chunk, topk, D):
    g = torch.Generator(device="cuda").manual_seed(L + D)
    mk = lambda h: torch.randn((L, h, D), generator=g, device="cuda").to(torch.bfloat16)
    q, k, v, dout, cu = mk(1), mk(1), mk(1), mk(1), torch.tensor([0, L], dtype=torch.int32, device="cuda")
    csc = flash_moba.flash_topk_varlen_func(q, k, cu, cu, L, L, topk, chunk, causal=True)
    out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, *csc, cu, cu, None, None, None, L, L, 0.0, D ** -0.5, False, True, 0.0, False, 128, chunk, None)
    dq, dk, dv, _ = hip.moba_varlen_bwd(dout, q, k, v, out, lse, None, None, None, *csc, cu, cu, None, L, L, 0.0, D ** -0.5, False, True, 0.0, False,
                                        128, chunk, None, _dq_mode=1)
    for name, x, y in zip(("dq", "dk", "dv"), (dq, dk, dv), _reference(q, k, v, dout, [0, L], *csc, chunk)[1:]):
        assert_close(name, x, y, 2e-2, 1e-2)  # (the bounds of the other attention tests)
