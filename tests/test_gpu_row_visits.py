"""Visits per (row, head) of a pattern and their maximum, counted from lists in any order."""
import ctypes

import numpy as np
import pytest
import torch

from flash_moba import flash_moba_hip as hip

pytestmark = pytest.mark.gpu


# Atomics in memory; ranges of rows that end inside a sequence, sequences of no rows, of one; more than
# 512 columns; lists of more than 512 entries, unequal in pairs; columns whose last key block is cut short; rows of no sequence
@pytest.mark.parametrize("lens_q,lens_k,heads,chunk,rest", [
    ([3000, 1, 0, 1025], [3000, 700, 64, 1025], 2, 64, 0), ([300, 90], [300, 90], 4, 192, 5), ([40000], [40000], 8, 64, 0),
    ([1500, 1500], [1500, 1700], 3, 128, 3), ([700], [1000], 1, 128, 1)])
def test_counts(lens_q, lens_k, heads, chunk, rest):
    rng = np.random.default_rng(sum(lens_q) + chunk)
    cols = -(-max(lens_k) // chunk)
    kb = 128 if chunk % 128 == 0 else 64
    total = sum(lens_q) + rest
    off, nnz, rows = np.zeros((len(lens_q), heads, cols), np.int64), np.zeros((len(lens_q), heads, cols), np.int32), []
    want, at, q0 = np.zeros((total, heads), np.int64), 0, 0
    for b, (nq, nk) in enumerate(zip(lens_q, lens_k)):
        for h in range(heads):
            for c in range(-(-nk // chunk)):
                n = int(rng.integers(0, min(nq, 1300) + 1)) if nq else 0
                r = rng.permutation(nq)[:n] if nq < 5000 else rng.integers(0, nq, n)
                off[b, h, c], nnz[b, h, c] = at, n
                at += n
                rows.append(r)
                np.add.at(want[:, h], q0 + r, -(-min(chunk, nk - c * chunk) // kb))
        q0 += nq
    dev = lambda x, t: torch.from_numpy(np.ascontiguousarray(x)).to(t).cuda()
    keep = [dev(off, torch.int64), dev(nnz, torch.int32), dev(np.concatenate(rows + [np.zeros(1)]), torch.int32),
            dev(np.cumsum([0] + lens_q), torch.int32), dev(np.cumsum([0] + lens_k), torch.int32)]
    a = hip.AttnFwdArgs()
    a.col_offsets, a.col_nnz, a.row_indices, a.cu_seqlens_q, a.cu_seqlens_k = (t.data_ptr() for t in keep)
    a.batch, a.total_q, a.total_k, a.heads, a.heads_k, a.head_dim = len(lens_q), total, sum(lens_k), heads, heads, 64
    a.max_seqlen_q, a.max_seqlen_k, a.max_cols, a.lg_block_m, a.lg_block_n, a.is_causal, a.dtype = max(lens_q), max(lens_k), cols, 128, chunk, 1, 1
    counts = torch.full((total * heads + 1,), -1, dtype=torch.int32, device="cuda")
    rc = hip.load_library().fmoba_csc_max_row_visits(ctypes.byref(a), counts.data_ptr(), counts[total * heads:].data_ptr(),
                                                     torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert np.array_equal(counts[:-1].cpu().numpy().reshape(total, heads), want) and int(counts[-1]) == want.max()


# the same counted in LDS: many pairs of the longest sequence's length, or lists that are short
@pytest.mark.parametrize("lens_q,lens_k,heads,chunk,rest", [
    ([3000, 1, 0, 1025] * 2, [3000, 700, 64, 1025] * 2, 8, 64, 0), ([300, 90] * 8, [300, 90] * 8, 4, 192, 5), ([40000], [40000], 12, 64, 0),
    ([1500, 1500] * 6, [1500, 1700] * 6, 3, 128, 3), ([300], [400], 8, 128, 1)])
def test_counts_in_lds(lens_q, lens_k, heads, chunk, rest):
    f = hip.AttnFwdArgs()
    f.heads, f.total_q, f.max_seqlen_q, f.max_cols = heads, sum(lens_q) + rest, max(lens_q), -(-max(lens_k) // chunk)
    assert hip.load_library().fmoba_csc_row_visits_in_lds(ctypes.byref(f)) == 1
    test_counts(lens_q, lens_k, heads, chunk, rest)
