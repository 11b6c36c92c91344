"""Selection words of a caller's own lists: sequences whose words fit a workgroup's LDS and longer ones, lists in any order."""
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip

pytestmark = pytest.mark.gpu


# the last length that fits, the first that does not; sequences of one row, of none, at both sizes of the workgroup; more than 32 chunks; lists
# of more entries than a turn of the waves takes, and empty ones
@pytest.mark.parametrize("lens,H,D,chunk", [([32768], 1, 64, 4096), ([32769], 1, 64, 4096), ([1, 0, 1024, 300], 3, 128, 64), ([1025, 5, 2500], 2, 96, 64)])
def test_rows_of_lists_in_any_order(lens, H, D, chunk):
    g = torch.Generator(device="cuda").manual_seed(sum(lens))
    C, T = -(-max(lens) // chunk), sum(lens)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
    co, cn = torch.zeros((len(lens), H, C), dtype=torch.int64, device="cuda"), torch.zeros((len(lens), H, C), dtype=torch.int32, device="cuda")
    lists, mixed, at, dense = [], [], 0, []
    for b, n in enumerate(lens):
        for h in range(H):
            c = torch.arange(C, device="cuda")[None]
            own = (torch.arange(n, device="cuda") // chunk)[:, None]
            sel = (c <= own) & ((c == own) | (c == 0) | (torch.rand((n, C), generator=g, device="cuda") < 0.6)) & (c != 2)
            dense.append(sel)
            for i in range(C):
                r = sel[:, i].nonzero().flatten().int()
                co[b, h, i], cn[b, h, i] = at, r.numel()
                lists.append(r), mixed.append(r[torch.randperm(r.numel(), generator=g, device="cuda")])
                at += r.numel()
    q, k, v = (torch.randn((T, H, D), generator=g, device="cuda").to(torch.bfloat16) for _ in range(3))

    def call(rows):
        with torch.no_grad():
            out = flash_moba.flash_moba_attn_varlen_func(q, k, v, cu, cu, max(lens), max(lens), co, cn, torch.cat(rows), lg_block_m=128, lg_block_n=chunk, causal=True)
        assert hip.last_fwd_row_blocks()
        return out

    got = call(lists)
    assert torch.equal(call(mixed), got)
    for b, n in enumerate(lens):  # against fp32, the rows that see the most
        for h in range(H):
            r = torch.arange(max(0, n - 64), n, device="cuda")
            if not n:
                continue
            s, x = int(cu[b]), [t[int(cu[b]):int(cu[b]) + n, h].float() for t in (q, k, v)]
            keep = dense[b * H + h][r].repeat_interleave(chunk, 1)[:, :n] & (torch.arange(n, device="cuda")[None] <= r[:, None])
            p = torch.softmax((x[0][r] @ x[1].T * D ** -0.5).masked_fill(~keep, float("-inf")), -1).nan_to_num(0.0)
            # P and the output rounded to 8 bits, each relative to sums of |P V| of about 1
            assert torch.allclose(got[s + r, h].float(), p @ x[2], atol=2e-2, rtol=2e-2)
