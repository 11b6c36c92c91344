"""dK and dV of query heads kept apart, added up over a group: every edge of a workgroup, any number of heads, any strides."""
import pytest
import torch

from flash_moba import flash_moba_hip as hip

pytestmark = pytest.mark.gpu


# no rows; less than a workgroup of vectors; a row that ends inside one; a row of more vectors than a workgroup has; groups of one, of no multiple of the unroll, of many
@pytest.mark.parametrize("rows,heads_k,grp,dim", [(0, 2, 4, 128), (1, 1, 2, 8), (3, 1, 64, 64), (37, 3, 5, 40), (129, 8, 4, 96), (515, 20, 1, 256), (1000, 2, 7, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", ["packed", "slices", "heads_first"])
def test_sums_of_groups(rows, heads_k, grp, dim, dtype, layout):
    g = torch.Generator().manual_seed(rows + dim)
    apart = torch.randn((2, rows, heads_k * grp, dim), generator=g).to(dtype).cuda()
    if layout == "packed":
        whole = torch.zeros((2, rows, heads_k, dim), dtype=dtype, device="cuda")
        dk, dv = whole[0], whole[1]
    elif layout == "slices":
        whole = torch.zeros((rows, 3, heads_k, dim), dtype=dtype, device="cuda")
        dk, dv = whole[:, 1], whole[:, 2]
    else:
        whole = torch.zeros((2, heads_k, rows, dim), dtype=dtype, device="cuda")
        dk, dv = whole[0].transpose(0, 1), whole[1].transpose(0, 1)
    hip._check(hip.load_library().fmoba_sum_grouped_heads(apart.data_ptr(), dk.data_ptr(), dv.data_ptr(), rows, heads_k * grp, heads_k, dim, dk.stride(0), dk.stride(1),
                                                          dv.stride(0), dv.stride(1), hip._dt(apart), hip._stream()))
    x = apart.cpu().double().view(2, rows, heads_k, grp, dim)
    ref, mass = x.sum(3), x.abs().sum(3)
    # one rounding to 16 bits of an fp32 sum of grp terms (half a unit in the last place of the result; below 2^-14 fp16 has steps of 2^-24)
    bound = ref.abs() * (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) + 2.0 ** -25 + mass * grp * 2.0 ** -23
    for got, r, b in ((dk, ref[0], bound[0]), (dv, ref[1], bound[1])):
        assert rows == 0 or ((got.cpu().double() - r).abs() <= b).all()
    if layout == "slices":
        assert not whole[:, 0].any()


def test_refusals():
    t = torch.zeros((2, 4, 4, 64), dtype=torch.bfloat16, device="cuda")
    lib = hip.load_library()
    call = lambda p=t.data_ptr(), heads=4, heads_k=2, dim=64, stride=64: lib.fmoba_sum_grouped_heads(p, t.data_ptr(), t.data_ptr(), 4, heads, heads_k, dim, 4 * 64, stride, 4 * 64, 64, hip._dt(t), hip._stream())
    for bad in (dict(p=None), dict(p=t.data_ptr() + 2), dict(heads=3), dict(heads_k=0), dict(dim=60), dict(stride=60)):
        assert call(**bad) != 0
