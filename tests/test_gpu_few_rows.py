"""Calls with at most eight query rows per sequence: their own gate and attention kernels."""
import numpy as np
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip
from flash_moba.mean_pool import flash_topk_mean_pool
from test_gpu_host_path import _both
from gpu_utils import assert_close
from oracle import moba_oracle as O

pytestmark = pytest.mark.gpu


def _case(lens_q, lens_k, H, Hk, D, dtype, seed, integer=False):
    g = torch.Generator().manual_seed(seed)
    mk = lambda n, h: (torch.randint(-2, 3, (n, h, D), generator=g).float() if integer else torch.randn((n, h, D), generator=g)).to(dtype)
    cu = lambda lens: torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32)
    return mk(sum(lens_q), H), mk(sum(lens_k), Hk), mk(sum(lens_k), Hk), cu(lens_q), cu(lens_k)


# chunks per sequence: none before the row's own, one tile of 32, at and past 64 and 256 (registers of a lane), past 1024;
# rows: one, eight, none; ties everywhere with integer inputs
@pytest.mark.parametrize("lens_q,lens_k,chunk,topk", [
    ([1], [5], 64, 3), ([1, 1, 0, 1], [2048, 64, 100, 65], 64, 4), ([8, 3], [64 * 65 + 1, 700], 64, 7), ([1, 2], [64 * 257, 64 * 40], 64, 33),
    ([4], [3000], 2, 16), ([1, 1], [4096, 2500], 1, 64), ([5], [3], 64, 2)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("integer", [True, False])
@pytest.mark.parametrize("D", [64, 96, 256])
def test_gate_selects_what_the_wide_gates_select(lens_q, lens_k, chunk, topk, causal, integer, D):
    # the same rows inside a longer query block go through the gates with 128 rows per workgroup
    q, k, _, cuq, cuk = (t.cuda() for t in _case(lens_q, lens_k, 4, 2, D, torch.bfloat16, len(lens_k) + topk, integer))
    mq, mk = max(lens_q), max(lens_k)
    km, cu_km, _ = flash_topk_mean_pool(k, cuk, mk, chunk)
    few = hip.moba_fused_topk(q, km, cuq, cuk, cu_km, mq, mk, topk, chunk, causal, return_raw=False, return_selection=True)
    wide = hip.moba_fused_topk(q, km, cuq, cuk, cu_km, 9, mk, topk, chunk, causal, return_raw=False, return_selection=True)
    assert all(torch.equal(few[i], wide[i]) for i in (0, 1, 2, 5))


@pytest.mark.parametrize("lens_q,lens_k,chunk,topk", [
    ([1], [5], 64, 3), ([1, 1, 1, 0, 1], [2048, 64, 129, 100, 3000], 128, 4), ([3, 8], [1000, 4097], 64, 5), ([1, 2], [64 * 257, 64 * 40], 256, 9)])
@pytest.mark.parametrize("H,Hk", [(4, 4), (8, 1)])
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (40, torch.float16), (128, torch.float16), (96, torch.bfloat16), (256, torch.bfloat16), (160, torch.float16)])
def test_attention_of_a_few_rows(lens_q, lens_k, chunk, topk, H, Hk, D, dtype):
    q, k, v, cuq, cuk = _case(lens_q, lens_k, H, Hk, D, dtype, D + topk)
    mq, mk = max(lens_q), max(lens_k)
    where = (cuq.cuda(), cuk.cuda(), mq, mk)
    out = flash_moba.flash_moba_varlen_func(q.cuda(), k.cuda(), v.cuda(), *where, chunk, topk, causal=True)
    co, cn, ind = flash_moba.flash_topk_varlen_func(q.cuda(), k.cuda(), *where, topk, chunk, causal=True)
    cols, lse, _, _ = hip.moba_varlen_fwd(q.cuda(), k.cuda(), v.cuda(), None, co, cn, ind, *where[:2], None, None, None, mq, mk, 0.0, D ** -0.5,
                                          False, True, 0.0, False, 128, chunk, None, _fwd_mode=1)
    out2, lse2, _, _ = hip.moba_varlen_fwd(q.cuda(), k.cuda(), v.cuda(), None, co, cn, ind, *where[:2], None, None, None, mq, mk, 0.0, D ** -0.5,
                                           False, True, 0.0, False, 128, chunk, None)
    assert torch.equal(out, out2)
    assert_close("out", out, cols.float().cpu(), 2e-2, 1e-2)
    assert_close("lse", lse2, lse.float().cpu(), 2e-3, 1e-3)


# scores that are infinite or not a number: a candidate needs a score above -inf, +inf comes first, ties go to the higher chunk
@pytest.mark.parametrize("lens_k,chunk,topk", [([2048, 700], 64, 5), ([64 * 257 + 3, 64 * 40], 64, 33), ([5000, 1500], 2, 16), ([2048, 900], 64, 64)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D", [64, 256])
def test_gate_with_infinite_scores_and_without_numbers(lens_k, chunk, topk, causal, D):
    lens_q, H, Hk = [3, 8], 4, 2
    q, k, _, cuq, cuk = (t.cuda() for t in _case(lens_q, lens_k, H, Hk, D, torch.bfloat16, topk, integer=True))
    km, cu_km, _ = flash_topk_mean_pool(k, cuk, max(lens_k), chunk)
    g = torch.Generator(device="cuda").manual_seed(topk)
    km.copy_(torch.randint(-2, 3, km.shape, generator=g, device="cuda"))
    q[:, :, 0] = torch.where(torch.rand(q.shape[:2], generator=g, device="cuda") < 0.5, 1.0, -1.0).to(q.dtype)
    kind = torch.randint(0, 8, km.shape[:2], generator=g, device="cuda")
    for i, special in enumerate((float("inf"), float("-inf"), float("nan"))):
        km[:, :, 0] = torch.where(kind == i, special, km[:, :, 0].float()).to(km.dtype)
    q[1] = float("nan")  # (a row without a score at all)
    words = hip.moba_fused_topk(q, km, cuq, cuk, cu_km, 8, max(lens_k), topk, chunk, causal, return_raw=False, return_selection=True)[5].cpu()
    C = -(-max(lens_k) // chunk)
    got = (words[:, torch.arange(C) // 32, :] >> (torch.arange(C) % 32)[None, :, None]) & 1  # heads, chunks, rows
    kpos = cu_km.cpu().tolist()
    row = 0
    for b, (nq, nk) in enumerate(zip(lens_q, lens_k)):
        for i in range(nq):
            pos = i + nk - nq
            n = pos // chunk if causal else kpos[b + 1] - kpos[b]
            for h in range(H):
                score = (km[kpos[b]:kpos[b] + n, h // (H // Hk)].double().cpu() @ q[row, h].double().cpu()).tolist()
                order = sorted((c for c in range(n) if score[c] > float("-inf")), key=lambda c: (-score[c], -c))
                want = set(order[:topk - 1] + [pos // chunk] if causal else order[:topk])
                assert set(got[h, :, row].nonzero().flatten().tolist()) == want, (b, i, h)
            row += 1


def _fwd_args(lens_q, lens_k, H, Hk, D, chunk, topk, causal=True):
    """The sizes of a call of flash_moba_varlen_func."""
    f = hip.AttnFwdArgs()
    f.batch, f.total_q, f.total_k, f.heads, f.heads_k, f.head_dim = len(lens_q), sum(lens_q), sum(lens_k), H, Hk, D
    f.max_seqlen_q, f.max_seqlen_k, f.max_cols, f.lg_block_m, f.lg_block_n = max(lens_q), max(lens_k), -(-max(lens_k) // chunk), 128, chunk
    f.is_causal, f.max_visits_per_row = int(causal and max(lens_q) != 1), topk * (chunk // hip.fwd_key_block(chunk))
    f.q_row_stride = f.o_row_stride = H * D
    f.k_row_stride = f.v_row_stride = Hk * D
    f.q_head_stride = f.k_head_stride = f.v_head_stride = f.o_head_stride = D
    return f


# Scores from the pooling pass and the choice in front of the attention, against the gate and the attention over its selection bits.  Chunks at and past
# a lane's registers (256, 1024), products full of rows (4 heads x 8 rows), ties, keys that are infinite or not a number, more key heads than a block has.
@pytest.mark.parametrize("lens_q,lens_k,chunk,topk", [
    ([1], [5], 64, 3), ([1, 1, 0, 1], [64 * 65, 64, 100, 129], 64, 1), ([8, 3], [64 * 65 + 1, 700], 64, 7), ([8, 3], [64 * 65 + 1, 900], 64, 7),
    ([1, 2], [64 * 257, 64 * 256], 64, 33), ([1, 1], [64 * 1024, 64 * 1025 + 9], 64, 64), ([2], [1], 128, 5), ([4, 1], [128 * 300, 128 * 7], 128, 16)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("kind", ["normal", "ties", "special"])
@pytest.mark.parametrize("H,Hk,D,dtype", [(8, 2, 128, torch.bfloat16), (10, 10, 64, torch.float16), (12, 3, 256, torch.bfloat16), (12, 6, 96, torch.float16),
                                          (6, 6, 40, torch.bfloat16)])
def test_scores_from_the_pooling_pass(monkeypatch, lens_q, lens_k, chunk, topk, causal, kind, H, Hk, D, dtype):
    # (calls whose rows share too much to be read one by one keep the launch of the gate)
    scored = hip.load_library().fmoba_attn_fwd_gated_few_bytes(_fwd_args(lens_q, lens_k, H, Hk, D, chunk, topk, causal)) > 0
    assert scored == (H == Hk or (H, Hk) == (12, 6) or lens_k not in ([64 * 65 + 1, 700], [1]))
    q, k, v, cuq, cuk = (t.cuda() for t in _case(lens_q, lens_k, H, Hk, D, dtype, D + topk, kind == "ties"))
    if kind == "special":
        g = torch.Generator(device="cuda").manual_seed(topk)
        at = torch.randint(0, 300, k.shape[:2], generator=g, device="cuda")
        for i, x in enumerate((float("inf"), float("-inf"), float("nan"))):
            k[:, :, 0] = torch.where(at == i, x, k[:, :, 0].float()).to(dtype)
    out = lambda: (flash_moba.flash_moba_varlen_func(q, k, v, cuq, cuk, max(lens_q), max(lens_k), chunk, topk, causal=causal).view(torch.int16),)
    _both(monkeypatch, out)


@pytest.mark.parametrize("heads,heads_k,dim,rows,takes", [(32, 8, 128, 1, True), (32, 8, 128, 8, True), (32, 4, 128, 8, False), (8, 8, 96, 1, True), (8, 8, 256, 8, True)])
def test_which_calls_the_pooling_pass_scores(heads, heads_k, dim, rows, takes):
    f = hip.AttnFwdArgs()
    f.batch, f.total_q, f.total_k, f.heads, f.heads_k, f.head_dim = 4, 4 * rows, 4 << 16, heads, heads_k, dim
    f.max_seqlen_q, f.max_seqlen_k, f.max_cols, f.lg_block_n, f.is_causal, f.max_visits_per_row = rows, 1 << 16, 512, 128, 1, 8
    assert (hip.load_library().fmoba_attn_fwd_gated_few_bytes(f) > 0) == takes


def test_the_entry_point_needs_no_place_for_chunk_means(monkeypatch):
    lens_q, lens_k, H, Hk, D, chunk, topk = [1, 2], [5000, 900], 8, 2, 128, 64, 5
    q, k, v, cuq, cuk = (t.cuda() for t in _case(lens_q, lens_k, H, Hk, D, torch.bfloat16, 5))
    f, lib, stream = _fwd_args(lens_q, lens_k, H, Hk, D, chunk, topk), hip.load_library(), torch.cuda.current_stream().cuda_stream
    f.dtype, f.softmax_scale = 1, D ** -0.5  # (bf16)
    out, lse = torch.empty_like(q), torch.empty((H, sum(lens_q)), device="cuda")
    scores = torch.empty(lib.fmoba_attn_fwd_gated_few_bytes(f), dtype=torch.uint8, device="cuda")
    cu_km = torch.empty_like(cuk)
    f.q, f.k, f.v, f.out, f.softmax_lse, f.cu_seqlens_q, f.cu_seqlens_k = (t.data_ptr() for t in (q, k, v, out, lse, cuq, cuk))
    m = hip.MeanPoolArgs(k=f.k, cu_seqlens_k=f.cu_seqlens_k, cu_seqlens_km=cu_km.data_ptr(), batch=f.batch, max_chunks=f.max_cols, heads_k=Hk, head_dim=D, chunk=chunk,
                         dtype=f.dtype, k_row_stride=f.k_row_stride, k_head_stride=D)
    assert lib.fmoba_attn_fwd_gated_few(m, f, topk, 1, scores.data_ptr(), stream) == 0, lib.fmoba_last_error()
    want = _both(monkeypatch, lambda: (flash_moba.flash_moba_varlen_func(q, k, v, cuq, cuk, max(lens_q), max(lens_k), chunk, topk, causal=True),))[0]
    assert torch.equal(out, want)
