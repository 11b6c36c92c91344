"""Backward into the caller's dK and dV where query heads that were kept apart are added up: any tensors of the right shape and a last dimension of consecutive elements."""
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip

pytestmark = pytest.mark.gpu


# a dimension of one element may have any stride, whatever is said about the others (one key head; one key); rows that start anywhere; rows of no multiple of eight elements
@pytest.mark.parametrize("layout", ["packed", "head_stride_1", "row_stride_1", "odd_start", "odd_rows"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_any_layout(layout, dtype):
    T, H, D, chunk, topk = (1 if layout == "row_stride_1" else 777), 8, 128, 64, 3
    g = torch.Generator(device="cuda").manual_seed(T)
    mk = lambda h: torch.randn((T, h, D), generator=g, device="cuda").to(dtype)
    q, k, v, dout = mk(H), mk(1), mk(1), mk(H)
    cu = torch.tensor([0, T], dtype=torch.int32, device="cuda")
    lists = flash_moba.flash_topk_varlen_func(q, k, cu, cu, T, T, topk, chunk, causal=True)
    scale = D ** -0.5
    out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, *lists, cu, cu, None, None, None, T, T, 0.0, scale, False, True, 0.0, False, 128, chunk, None)

    def place():
        if layout == "packed":
            return torch.empty((T, 1, D), dtype=dtype, device="cuda")
        if layout == "head_stride_1":
            return torch.empty((T, D, 1), dtype=dtype, device="cuda").transpose(1, 2)
        if layout == "row_stride_1":
            return torch.empty((D,), dtype=dtype, device="cuda").as_strided((1, 1, D), (1, 1, 1))
        if layout == "odd_start":
            return torch.empty((T * D + 1,), dtype=dtype, device="cuda")[1:].view(T, 1, D)
        return torch.empty((T, 1, D + 3), dtype=dtype, device="cuda")[..., :D]

    run = lambda dk, dv: hip.moba_varlen_bwd(dout, q, k, v, out, lse, None, dk, dv, *lists, cu, cu, None, T, T, 0.0, scale, False, True, 0.0, False, 128, chunk)
    want = run(None, None)
    dk, dv = place(), place()
    got = run(dk, dv)
    assert got[1] is dk and got[2] is dv
    for a, b in zip(got, want):
        # a sum of eight heads in fp32 in another order, rounded once: at most one step of the 16-bit result apart
        assert (a.float() - b.float()).abs().max() <= (2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -10) * b.float().abs().max()
