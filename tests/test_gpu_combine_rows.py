"""Sums of a row's partial results: numbers of visits around every step of them, over plain and ranked lists, with NaN in what no visit wrote."""
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip

pytestmark = pytest.mark.gpu


# four (two) rows at a time, sixteen headers at a time; the first rows of the sequence have fewer visits than any of these
@pytest.mark.parametrize("topk", [1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 20, 31, 33])
@pytest.mark.parametrize("D", [40, 64, 128, 200])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_number_of_visits(topk, D, dtype):
    lens, H, Hk, chunk = [2400, 70, 1], 2, 1, 64
    T, L, scale = sum(lens), max(lens), D ** -0.5
    g = torch.Generator(device="cuda").manual_seed(topk + D)
    mk = lambda h: torch.randn((T, h, D), generator=g, device="cuda").to(dtype)
    q, k, v, dout = mk(H), mk(Hk), mk(Hk), mk(H)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
    plain = list(flash_moba.flash_topk_varlen_func(q, k, cu, cu, L, L, topk, chunk, causal=True))
    *ranked, selection, visits = hip.pool_and_gate_ranked(q, k, cu, cu, L, L, topk, chunk, True)

    def run(lists, fwd_mode, dq_mode, **kw):
        torch.full((T * H * topk * 260,), float("nan"), device="cuda")  # what the workspace is made of next
        out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, *lists, cu, cu, None, None, None, L, L, 0.0, scale, False, True, 0.0, False, 128, chunk, None, _fwd_mode=fwd_mode,
                                             _max_visits=topk, **kw)
        dq = None
        if D <= 128:
            dq = hip.moba_varlen_bwd(dout, q, k, v, out, lse, None, None, None, *lists, cu, cu, None, L, L, 0.0, scale, False, True, 0.0, False, 128, chunk, None,
                                     _dq_mode=dq_mode, _max_visits=topk, **kw)[0]
        return out, lse, dq

    want, want_lse, want_dq = run(plain, 2, 1)
    assert hip.last_fwd_row_blocks() == 1
    columns = [run(plain, 1, 2), run(ranked, 1, 2, _visits=visits)]
    assert hip.last_fwd_row_blocks() == 0
    step = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for out, lse, dq in columns:
        # probabilities and results are rounded to 16 bits in both, partial rows in one of them
        assert (out.float() - want.float()).norm() <= 2 * step * want.float().norm()
        assert (out.float() - want.float()).abs().max() <= 4 * step * v.float().abs().max()
        assert (lse - want_lse).abs().max() <= 1e-5 * want_lse.abs().max()
        if dq is not None:
            # half a step of each partial row: independent, so about half a step of their sum; at one element a few times the mean
            assert (dq.float() - want_dq.float()).norm() <= 2 * step * want_dq.float().norm()
            assert (dq.float() - want_dq.float()).abs().max() <= 4 * step * want_dq.float().abs().max()
    for a, b in zip(*columns):
        assert a is None or torch.equal(a, b)  # key order in both
