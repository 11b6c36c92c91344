"""Partial results of the column passes: their precision and their range against exact sums in 64 bits."""
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip

pytestmark = pytest.mark.gpu

# half a unit in the last place of the output, relative to the value, and the 32-bit sums under it
_HALF_ULP = {torch.bfloat16: 2.0 ** -8 * (1 + 2 ** -6), torch.float16: 2.0 ** -11 * (1 + 2 ** -6)}


def _uniform_rows(L, H, D, dtype, size, seed=0):
    """Equal scores (q = 0): every probability is exactly 1 before it is normalised, and row i of a causal call that sees all
    chunks is the mean of v[: i + 1]."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    q = torch.zeros((L, H, D), device="cuda", dtype=dtype)
    k = torch.randn((L, H, D), generator=g, device="cuda").to(dtype)
    v = (size * (1 + 0.5 * torch.rand((L, H, D), generator=g, device="cuda"))).to(dtype)
    exact = v.double().cumsum(0) / torch.arange(1, L + 1, device="cuda", dtype=torch.float64)[:, None, None]
    return q, k, v, torch.tensor([0, L], dtype=torch.int32, device="cuda"), exact


# above head dimension 128 the sums of a row are fp32 from end to end: a result is rounded once
@pytest.mark.parametrize("dtype,size", [(torch.bfloat16, 1.0), (torch.float16, 1.0), (torch.float16, 2000.0)])
@pytest.mark.parametrize("D", [136, 192, 256])
@pytest.mark.parametrize("chunk", [64, 128])
def test_wide_heads_round_once(dtype, size, D, chunk):
    L = 900
    q, k, v, cu, exact = _uniform_rows(L, 2, D, dtype, size, D)
    out = flash_moba.flash_moba_varlen_func(q, k, v, cu, cu, L, L, chunk, 15, causal=True)
    assert hip.last_fwd_row_blocks() == 0
    assert ((out.double() - exact).abs() <= _HALF_ULP[dtype] * exact).all()


# fp16 rows of the column form: up to 128 equal probabilities times values of 2000 are beyond the type, the results are not
@pytest.mark.parametrize("D", [40, 64, 128])
@pytest.mark.parametrize("chunk", [64, 128])
@pytest.mark.parametrize("size", [2.0 ** -13, 1.0, 2000.0, 40000.0])
def test_fp16_column_rows_keep_to_their_range(D, chunk, size):
    L = 900
    q, k, v, cu, exact = _uniform_rows(L, 2, D, torch.float16, size, D)
    co, cn, ind = flash_moba.flash_topk_varlen_func(q, k, cu, cu, L, L, 15, chunk, causal=True)
    out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, co, cn, ind, cu, cu, None, None, None, L, L, 0.0, 1.0, False, True, 0.0, False, 128, chunk, None,
                                         _fwd_mode=1)
    # a partial row and the result are rounded once each; values below 2^-14 have a fixed step of 2^-24
    tol = 2 * _HALF_ULP[torch.float16] * exact + 2.0 ** -24
    assert ((out.double() - exact).abs() <= tol).all()
    n = torch.arange(1, L + 1, device="cuda", dtype=torch.float64)
    assert ((lse.double() - n.log()).abs() <= 1e-5).all()


# fp16 partial rows of dQ: 64 keys of one sign add up to several times 65504 before the softmax scale, not after it
@pytest.mark.parametrize("D,chunk", [(64, 64), (40, 128), (96, 64), (128, 64), (128, 128)])
@pytest.mark.parametrize("scale", [None, 2.0])  # (a scale above one must not take range away either)
def test_fp16_dq_partial_rows_keep_to_their_range(D, chunk, scale):
    L, H = 300, 2
    val = 2000.0 if scale is None else 100.0
    scale = scale or D ** -0.5
    g = torch.Generator(device="cuda").manual_seed(D)
    s = (torch.randint(0, 2, (L, H, 1), generator=g, device="cuda") * 2 - 1).half()
    q, k, v = torch.zeros((L, H, D), device="cuda").half(), (2 * s).expand(L, H, D).contiguous(), (val * s).expand(L, H, D).contiguous()
    dout = torch.ones_like(q)
    cu = torch.tensor([0, L], dtype=torch.int32, device="cuda")
    co, cn, ind = flash_moba.flash_topk_varlen_func(q, k, cu, cu, L, L, 5, chunk, causal=True)
    csc = (co, cn, ind, cu, cu)
    out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, *csc, None, None, None, L, L, 0.0, scale, False, True, 0.0, False, 128, chunk, None)
    dq, _, _, _ = hip.moba_varlen_bwd(dout, q, k, v, out, lse, None, None, None, *csc, None, L, L, 0.0, scale, False, True, 0.0, False, 128, chunk, None,
                                      _dq_mode=2)
    # P = 1 / n over the row's n keys, m the mean sign: dq = scale * sum_j (dP_j - delta) K_j / n, dP_j = val D s_j, delta = val D m
    n = torch.arange(1, L + 1, device="cuda", dtype=torch.float64)[:, None, None]
    m = s.double().cumsum(0) / n
    size = scale * val * D * 2
    exact = (size * (1 - m * m)).expand(L, H, D)
    assert exact.max() < 65504 and exact.max() > 0.9 * size
    # Rows of fewer than 8 keys are left out: dS itself, 16-bit in every form, is up to val D 2 / n, beyond 65504 for them.
    # Roundings of out (in delta), P, dS, up to five partial rows and the result, each 2^-11 of at most `size`
    assert ((dq.double() - exact)[7:].abs() <= 9 * 2.0 ** -11 * size).all()


@pytest.mark.parametrize("D", [136, 256])
@pytest.mark.parametrize("chunk", [8192, 64 * 129])
def test_wide_heads_with_chunks_far_longer_than_the_sequence(D, chunk):
    q, k, v, cu, exact = _uniform_rows(500, 2, D, torch.bfloat16, 1.0, D)
    out = flash_moba.flash_moba_varlen_func(q, k, v, cu, cu, 500, 500, chunk, 64, causal=True)
    assert ((out.double() - exact).abs() <= _HALF_ULP[torch.bfloat16] * exact).all()


# both widths of a key block above head dimension 128 (eight waves for 128 keys, four for 64) against the row-block form: lists shorter
# than a tile and than a wave each, uneven tails, heads of a group in one workgroup
@pytest.mark.parametrize("D,dtype", [(136, torch.bfloat16), (192, torch.float16), (256, torch.bfloat16)])
@pytest.mark.parametrize("chunk,topk", [(64, 3), (128, 2), (128, 6), (192, 2), (256, 2)])
@pytest.mark.parametrize("H,Hk", [(2, 2), (6, 2), (8, 1)])
def test_wide_columns_against_row_blocks(D, dtype, chunk, topk, H, Hk):
    lens = [1, 0, 127, 129, 33, 1200]
    T, L = sum(lens), max(lens)
    g = torch.Generator(device="cuda").manual_seed(D + chunk + H)
    q, k, v = (torch.randn((T, h, D), generator=g, device="cuda").to(dtype) for h in (H, Hk, Hk))
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
    co, cn, ind = flash_moba.flash_topk_varlen_func(q, k, cu, cu, L, L, topk, chunk, causal=True)
    run = lambda form: hip.moba_varlen_fwd(q, k, v, None, co, cn, ind, cu, cu, None, None, None, L, L, 0.0, D ** -0.5, False, True, 0.0, False, 128, chunk,
                                           None, _fwd_mode=form)[:2]
    (out, lse), (want, want_lse) = run(1), run(2)
    # probabilities (relative to different maxima) and results are rounded to 16 bits in both
    step = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert (out.float() - want.float()).norm() <= step * want.float().norm()
    assert (out.float() - want.float()).abs().max() <= 4 * step * v.float().abs().max()
    assert (lse - want_lse).abs().max() <= 1e-5 * want_lse.abs().max()
    again = run(1)
    assert torch.equal(again[0], out) and torch.equal(again[1], lse)
