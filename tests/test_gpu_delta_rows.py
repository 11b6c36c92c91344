"""dot(dO, O) of every row, where the padded layout puts it, and zeros between the sequences."""
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip

pytestmark = pytest.mark.gpu


# fewer lanes to a row than rows to a lane (heads of 8 and 16) and more; sequences that end inside a lane's rows, inside a workgroup's and at their ends; output rows too
# many for the caches (64 MB and a little more) and a little fewer
@pytest.mark.parametrize("lens,H,D", [([1, 0, 63, 64, 65, 130, 2, 259], 3, d) for d in (8, 16, 24, 40, 64, 80, 128, 200, 256)] + [([5, 65531 + 3], 4, 128), ([5, 65531 - 9], 4, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_delta_of_every_row(lens, H, D, dtype):
    T, L, chunk = sum(lens), max(lens), 64 if max(lens) < 4096 else 4096
    g = torch.Generator(device="cuda").manual_seed(D)
    mk = lambda: torch.randn((T, H, D), generator=g, device="cuda").to(dtype)
    q, k, v, out, dout = mk(), mk(), mk(), mk(), mk()
    starts = [0] + torch.tensor(lens).cumsum(0).tolist()
    cu = torch.tensor(starts, dtype=torch.int32, device="cuda")
    lists = flash_moba.flash_topk_varlen_func(q, k, cu, cu, L, L, 1, chunk, causal=True)
    lse = torch.zeros((H, T), device="cuda")
    torch.full((H * (T + 128 * len(lens)),), float("nan"), device="cuda")  # what the result is made of next
    got = hip.moba_varlen_bwd(dout, q, k, v, out, lse, None, None, None, *lists, cu, cu, None, L, L, 0.0, 0.0, False, True, 0.0, False, 128, chunk)[3]
    prod = out.double() * dout.double()
    want, bound = (torch.zeros((H, T + 128 * len(lens)), dtype=torch.float64, device="cuda") for _ in range(2))
    for b, n in enumerate(lens):
        to = slice(starts[b] + 128 * b, starts[b] + 128 * b + n)
        want[:, to] = prod[starts[b]:starts[b + 1]].sum(-1).t()
        bound[:, to] = prod[starts[b]:starts[b + 1]].abs().sum(-1).t() * 2.0 ** -23 * 16  # eight products in a lane, then a tree over 32 lanes at most
    assert ((got.double() - want).abs() <= bound).all()
