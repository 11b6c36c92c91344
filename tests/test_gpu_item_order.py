"""Calls of few workgroups: the order of the work items, the split of a group's heads, the form of dQ.  Every item has to be taken once."""
import numpy as np
import pytest
import torch

import flash_moba
from gpu_utils import assert_close

pytestmark = pytest.mark.gpu


def _reference(q, k, v, dout, cu, col_offsets, col_nnz, rows, chunk):
    """out, dq, dk, dv of the pattern in fp32, a head at a time."""
    q, k, v, dout = (t.float() for t in (q, k, v, dout))
    H, grp, D = q.shape[1], q.shape[1] // k.shape[1], q.shape[2]
    off, nnz, rows = col_offsets.cpu().view(len(cu) - 1, H, -1), col_nnz.cpu().view(len(cu) - 1, H, -1), rows
    out, dq, dk, dv = torch.zeros_like(q), torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
    for b in range(len(cu) - 1):
        s, n = cu[b], cu[b + 1] - cu[b]
        for h in range(H):
            mask = torch.zeros(n, n, dtype=torch.bool, device="cuda")
            for c in range(-(-n // chunk)):
                lo = int(off[b, h, c])
                mask[rows[lo:lo + int(nnz[b, h, c])].long(), c * chunk:(c + 1) * chunk] = True
            mask &= torch.ones(n, n, dtype=torch.bool, device="cuda").tril()
            x, y, z, g = q[s:s + n, h], k[s:s + n, h // grp], v[s:s + n, h // grp], dout[s:s + n, h]
            p = torch.softmax((x @ y.T * D ** -0.5).masked_fill(~mask, float("-inf")), -1)
            out[s:s + n, h] = p @ z
            ds = p * (g @ z.T - (g * out[s:s + n, h]).sum(-1, keepdim=True)) * D ** -0.5
            dq[s:s + n, h] = ds @ y
            dk[s:s + n, h // grp] += ds.T @ x
            dv[s:s + n, h // grp] += p.T @ g
    return out, dq, dk, dv


# lengths at the edges of 256-row blocks; pairs that are a multiple of eight (odd and even multiples) and not; more items than one
# per unit but no more than two (the reversed second half of the dQ pass: 35 blocks of one pair per XCD, 17 of two, 32 and 33
# of one each side of the line); key heads shared by four and by eight
@pytest.mark.parametrize("lens,H,Hk,D,chunk,topk", [
    ([255, 256, 257], 8, 8, 128, 64, 2), ([1, 0, 513, 300], 4, 1, 64, 64, 3), ([700, 40], 3, 3, 128, 64, 2),
    ([700, 1, 130, 513], 8, 1, 96, 128, 2), ([1025], 16, 2, 128, 128, 2), ([1025], 8, 1, 64, 64, 2),
    ([300] * 33, 8, 8, 128, 64, 3), ([4200], 16, 4, 128, 64, 20), ([8192], 8, 8, 128, 64, 26), ([8257], 8, 8, 128, 64, 26)])
def test_every_item_once(lens, H, Hk, D, chunk, topk):
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + D)
    mk = lambda h: torch.randn((sum(lens), h, D), generator=g, device="cuda").to(torch.bfloat16)
    q, k, v, dout = (x.requires_grad_(True) for x in (mk(H), mk(Hk), mk(Hk), mk(H)))
    cu = [0] + [int(x) for x in np.cumsum(lens)]
    cud = torch.tensor(cu, dtype=torch.int32, device="cuda")
    out = flash_moba.flash_moba_varlen_func(q, k, v, cud, cud, max(lens), max(lens), chunk, topk, causal=True)
    got = (out.detach(), *torch.autograd.grad(out, (q, k, v), dout.detach()))
    pattern = flash_moba.flash_topk_varlen_func(q.detach(), k.detach(), cud, cud, max(lens), max(lens), topk, chunk, causal=True)
    # (the bounds of the other attention tests: 16-bit results of sums of 16-bit factors; dk and dv add up the heads of a group, each with
    # an error of its own within the bound, so theirs is the group's sum of it)
    want = _reference(q.detach(), k.detach(), v.detach(), dout.detach(), cu, *pattern, chunk)
    for name, x, y, n in zip(("out", "dq", "dk", "dv"), got, want, (1, 1, H // Hk, H // Hk)):
        assert_close(name, x, y, 2e-2 * n, 1e-2)
