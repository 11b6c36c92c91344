"""Gate over groups of 64 chunks (more than 128 chunks per sequence, at most 16 winners): scores that are exact, so the selection is known."""
import numpy as np
import pytest
import torch

import flash_moba
from gpu_utils import csc_selection_one_head

pytestmark = pytest.mark.gpu


def _scores(kind, C, D, g):
    """Key rows (C, D), each a chunk's mean; a query row e_d scores column d."""
    c = torch.arange(C).float()[:, None]
    if kind == "random":
        k = torch.randn((C, D), generator=g)
    elif kind == "levels":  # ties across every cut, zeros of both signs
        k = torch.randint(-2, 3, (C, D), generator=g).float() * 0.5
        k[(k == 0) & (torch.rand((C, D), generator=g) < 0.5)] = -0.0
    elif kind == "equal":
        k = torch.full((C, D), -3.0)
    elif kind == "ascending":  # every chunk is a winner when it comes
        k = c - C // 2 + torch.zeros(1, D)
    else:  # "descending", with large values among them (their chunk sums stay finite)
        k = C // 2 - c + torch.zeros(1, D)
        k[3], k[C // 2] = 2.0 ** 124, -(2.0 ** 124)
    return k


# more than 128 chunks (the first group at most full, three groups and a rest, exact groups), more than 256; no winner, one, as many
# as the weak half of the places holds and one more, all sixteen; heads of 40 to 256; the causal rule and the plain one
@pytest.mark.parametrize("kind", ["random", "levels", "equal", "ascending", "descending"])
@pytest.mark.parametrize("C,topk,D,causal", [
    (129, 9, 64, True), (192, 10, 128, True), (200, 17, 40, True), (256, 1, 128, True), (255, 2, 256, True), (193, 16, 128, False),
    (321, 8, 128, False), (257, 16, 64, True), (640, 17, 128, True), (700, 9, 256, False)])
def test_selection_of_exact_scores(kind, C, topk, D, causal):
    chunk, H = 4, 2
    g = torch.Generator().manual_seed(C + topk)
    Lk = C * chunk - 1
    Lq = Lk if C in (129, 257) else 700
    off = Lk - Lq
    keys = [_scores(kind, C, D, g).to(torch.bfloat16) for _ in range(H)]
    k = torch.stack([x.repeat_interleave(chunk, 0)[:Lk] for x in keys], 1)
    pick = torch.randint(0, D, (Lq, H), generator=g)
    q = torch.nn.functional.one_hot(pick, D).to(torch.bfloat16)
    # infinite, undefined and negated scores in some rows
    special = torch.randint(0, 8, (Lq, H), generator=g)
    factor = torch.where(special == 0, float("inf"), torch.where(special == 1, float("nan"), torch.where(special == 2, -1.0, 1.0)))
    q = torch.where(q > 0, factor[..., None].to(torch.bfloat16), torch.zeros((), dtype=torch.bfloat16))
    cq, ck = (torch.tensor([0, n], dtype=torch.int32, device="cuda") for n in (Lq, Lk))
    co, cn, ind = flash_moba.flash_topk_varlen_func(q.cuda(), k.cuda(), cq, ck, Lq, Lk, topk, chunk, causal=causal)
    for h in range(H):
        score = (keys[h].double()[:, pick[:, h]] * factor[:, h].double()).T.numpy()  # (Lq, C); the other products are zeros
        got = csc_selection_one_head(co, cn, ind, 0, h, Lq).cpu().numpy()
        want = np.zeros((Lq, C), dtype=bool)
        for r in range(Lq):
            own = (r + off) // chunk
            n, kp = (own, topk - 1) if causal else (C, topk)
            cand = np.nonzero(score[r, :n] > -np.inf)[0]
            want[r, cand[np.lexsort((cand, score[r, cand]))][::-1][:kp]] = True
            if causal:
                want[r, own] = True
        assert (got == want).all(), np.argwhere(got != want)[:4]


def test_more_row_blocks_than_the_second_dimension_of_a_grid():
    L, chunk = 65536 * 128 + 5, 65536
    g = torch.Generator(device="cuda").manual_seed(0)
    x = torch.randn((L, 1, 8), generator=g, device="cuda").to(torch.bfloat16)
    cu = torch.tensor([0, L], dtype=torch.int32, device="cuda")
    co, cn, ind = flash_moba.flash_topk_varlen_func(x, x, cu, cu, L, L, 2, chunk, causal=True)
    off, nnz = co.flatten().tolist(), cn.flatten().tolist()
    rows = torch.zeros(L, dtype=torch.int32, device="cuda")
    for c in range(len(nnz)):
        e = ind[off[c]:off[c] + nnz[c]].long()
        own = torch.arange(c * chunk, min(L, (c + 1) * chunk), device="cuda")
        assert torch.equal(e[:own.numel()], own) and (e[1:] > e[:-1]).all()
        rows.index_add_(0, e, torch.ones_like(e, dtype=torch.int32))
    assert (rows[:chunk] == 1).all() and (rows[chunk:] == 2).all()


# the same with 16 and 32 places per lane: the first count beyond those of 8 and 16, the weak half full and one more, all places; fewer chunks
# than winners in the first group, and than winners at all in most rows
@pytest.mark.parametrize("kind", ["random", "levels", "equal", "ascending", "descending"])
@pytest.mark.parametrize("C,topk,D,causal", [
    (257, 18, 128, True), (300, 17, 64, False), (321, 33, 128, True), (260, 32, 256, False), (400, 34, 64, True), (290, 33, 128, False),
    (333, 64, 128, True), (520, 64, 40, False), (280, 64, 256, True), (257, 33, 64, True)])
def test_selection_of_exact_scores_with_many_winners(kind, C, topk, D, causal):
    test_selection_of_exact_scores(kind, C, topk, D, causal)
