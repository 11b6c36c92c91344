"""Gate of up to 128 chunks that takes a row's best scores off one by one (at most ten of them) or bisects: scores that are exact, so the selection is known."""
import numpy as np
import pytest
import torch

import flash_moba
from gpu_utils import csc_selection_one_head
from test_gpu_grouped_gate import _scores

pytestmark = pytest.mark.gpu


# fewer candidates than winners, one more, a tile of 32 and one more, both tiles, three and four; one winner, ten (the last count that is taken off) and eleven;
# ties across the cut, infinite and undefined scores
@pytest.mark.parametrize("kind", ["random", "levels", "equal", "ascending", "descending"])
@pytest.mark.parametrize("C,topk,D,causal", [(5, 2, 64, True), (12, 11, 64, True), (32, 5, 128, True), (33, 11, 40, True), (33, 1, 64, False), (64, 10, 64, False), (64, 12, 128, True),
                                             (65, 11, 96, True), (96, 3, 128, False), (128, 11, 256, True), (128, 11, 64, False)])
def test_selection_of_exact_scores(kind, C, topk, D, causal):
    chunk, H = 4, 2
    g = torch.Generator().manual_seed(C + topk)
    L = C * chunk - 1
    keys = [_scores(kind, C, D, g).to(torch.bfloat16) for _ in range(H)]
    k = torch.stack([x.repeat_interleave(chunk, 0)[:L] for x in keys], 1)
    pick = torch.randint(0, D, (L, H), generator=g)
    special = torch.randint(0, 8, (L, H), generator=g)
    factor = torch.where(special == 0, float("inf"), torch.where(special == 1, float("nan"), torch.where(special == 2, -1.0, 1.0)))
    q = torch.where(torch.nn.functional.one_hot(pick, D) > 0, factor[..., None].to(torch.bfloat16), torch.zeros((), dtype=torch.bfloat16))
    cu = torch.tensor([0, L], dtype=torch.int32, device="cuda")
    co, cn, ind = flash_moba.flash_topk_varlen_func(q.cuda(), k.cuda(), cu, cu, L, L, topk, chunk, causal=causal)
    for h in range(H):
        score = (keys[h].double()[:, pick[:, h]] * factor[:, h].double()).T.numpy()  # (L, C); the other products are zeros
        got = csc_selection_one_head(co, cn, ind, 0, h, L).cpu().numpy()
        want = np.zeros((L, C), dtype=bool)
        for r in range(L):
            own = r // chunk
            n, kp = (own, topk - 1) if causal else (C, topk)
            cand = np.nonzero(score[r, :n] > -np.inf)[0]
            want[r, cand[np.lexsort((cand, score[r, cand]))][::-1][:kp]] = True
            if causal:
                want[r, own] = True
        assert (got == want).all(), np.argwhere(got != want)[:4]
