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
