"""Partial rows of head dimensions that do not fill whole 64-byte pieces: padded, and what lies in the padding reaches no result."""
import numpy as np
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip
from gpu_utils import assert_close
from test_gpu_item_order import _reference

pytestmark = pytest.mark.gpu


# one 8-element piece past a whole 64 bytes, one before it, a whole number; rows of 16 bits and (above 128) of fp32; both key block sizes; lists with
# ranks and plain ones; a value column of infinities that the padding may hold copies of
@pytest.mark.parametrize("D", [8, 40, 56, 64, 72, 88, 96, 104, 120, 128, 136, 248])
@pytest.mark.parametrize("chunk", [64, 128])
@pytest.mark.parametrize("ranked", [False, True])
def test_partial_rows(D, chunk, ranked):
    L, H, topk = 1100, 2, 3
    g = torch.Generator(device="cuda").manual_seed(D + chunk)
    q, k, v, dout = (torch.randn((L, H, D), generator=g, device="cuda").to(torch.bfloat16) for _ in range(4))
    cu = torch.tensor([0, L], dtype=torch.int32, device="cuda")
    pattern = flash_moba.flash_topk_varlen_func(q, k, cu, cu, L, L, topk, chunk, causal=True)
    want = _reference(q, k, v, dout, [0, L], *pattern, chunk)
    if ranked:  # (the fused call chooses the form by itself: wide heads of this density go by columns)
        leaf = [t.clone().requires_grad_(True) for t in (q, k, v)]
        out = flash_moba.flash_moba_varlen_func(*leaf, cu, cu, L, L, chunk, topk, causal=True)
        got = (out.detach(), *torch.autograd.grad(out, leaf, dout))
    else:
        out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, *pattern, cu, cu, None, None, None, L, L, 0.0, D ** -0.5, False, True, 0.0, False, 128, chunk, None,
                                             _fwd_mode=1)
        assert hip.last_fwd_row_blocks() == 0
        got = (out, *hip.moba_varlen_bwd(dout, q, k, v, out, lse, None, None, None, *pattern, cu, cu, None, L, L, 0.0, D ** -0.5, False, True, 0.0, False,
                                         128, chunk, None, _dq_mode=2 if D <= 128 else 1)[:3])
    for name, x, y in zip(("out", "dq", "dk", "dv"), got, want):
        assert_close(name, x, y, 2e-2, 1e-2)  # (the bounds of the other attention tests)
    # an infinite value in the last feature alone: the other features, and the padding's neighbours, stay what they are
    v = v.clone()
    v[:, :, D - 1] = float("inf")
    inf = hip.moba_varlen_fwd(q, k, v, None, *pattern, cu, cu, None, None, None, L, L, 0.0, D ** -0.5, False, True, 0.0, False, 128, chunk, None, _fwd_mode=1)[0]
    assert not torch.isfinite(inf[..., D - 1]).any()  # (keys of the block that the row does not see have probability zero: 0 * inf)
    assert_close("out", inf[..., :D - 1], want[0][..., :D - 1], 2e-2, 1e-2)
