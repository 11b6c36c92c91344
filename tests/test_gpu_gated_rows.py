"""The row-block forward that chooses its rows' chunks itself (native host path) against gate and attention as two launches (path through the ops): same bits."""
import numpy as np
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip
from test_gpu_few_rows import _fwd_args
from test_gpu_host_path import _both

pytestmark = pytest.mark.gpu


# One row block and many; two waves and four, one set, two and four; one chunk, a tile of 32 and one more, 64; rows at the edges of a wave's 32 and a block's 64 and 128; queries that are the
# last rows of longer keys or come before the keys begin; empty sequences; heads of a group
@pytest.mark.parametrize("lens_q,lens_k,H,Hk,D,chunk,topk", [
    ([9], [9], 2, 2, 64, 64, 1), ([1024, 2048], [1024, 2048], 8, 8, 64, 128, 4), ([2048], [2048], 4, 2, 64, 64, 9), ([33, 0, 65, 300], [33, 7, 65, 300], 2, 1, 40, 64, 2),
    ([341] * 30, [341] * 30, 16, 16, 64, 64, 4), ([4096], [4096], 16, 16, 64, 64, 24), ([129, 2112], [129, 2112], 4, 4, 128, 64, 12), ([512, 90], [2049, 4000], 4, 4, 120, 64, 20),
    ([4096, 100], [4096, 100], 16, 4, 128, 64, 30), ([700], [300], 2, 2, 128, 64, 3),
    ([2048], [2048], 16, 4, 256, 64, 16), ([2000, 77], [2000, 77], 16, 16, 136, 64, 20)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("kind", ["normal", "ties", "special"])
@pytest.mark.parametrize("grad", [True, False])
def test_rows_that_choose_their_chunks(monkeypatch, lens_q, lens_k, H, Hk, D, chunk, topk, causal, kind, grad):
    # (without a causal limit 4 of 16 chunks are few: by columns)
    f, b = _fwd_args(lens_q, lens_k, H, Hk, D, chunk, topk, causal), hip.AttnBwdArgs()
    for name in ("batch", "total_q", "total_k", "heads", "heads_k", "head_dim", "max_seqlen_q", "max_seqlen_k", "max_cols", "lg_block_n", "is_causal"):
        setattr(b, name, getattr(f, name))
    b.max_visits_per_row = topk * (chunk // 64)
    assert hip.load_library().fmoba_attn_fwd_gates_rows(f) == (causal or lens_q != [1024, 2048])
    assert not hip.load_library().fmoba_attn_bwd_uses_partials(b)  # (whose lists are ranked by a gate of its own)
    g = torch.Generator(device="cuda").manual_seed(sum(lens_q) + D)
    dtype = torch.float16 if H == 4 else torch.bfloat16
    draw = (lambda s: torch.randint(-2, 3, s, generator=g, device="cuda").float()) if kind == "ties" else (lambda s: torch.randn(s, generator=g, device="cuda"))
    mk = lambda n, h: draw((n, h, D)).to(dtype)
    q, k, v, dout = mk(sum(lens_q), H), mk(sum(lens_k), Hk), mk(sum(lens_k), Hk), mk(sum(lens_q), H)
    if kind == "special":
        q[-3, 0], q[-7, 0] = float("inf"), float("nan")
        k[sum(lens_k) // 2, 0], k[sum(lens_k) // 3, -1] = float("inf"), float("nan")
    cq, ck = (torch.tensor([0] + list(np.cumsum(x)), dtype=torch.int32, device="cuda") for x in (lens_q, lens_k))

    def run():
        qg, kg, vg = (t.clone().requires_grad_(grad) for t in (q, k, v))
        out = flash_moba.flash_moba_varlen_func(qg, kg, vg, cq, ck, max(lens_q), max(lens_k), chunk, topk, causal=causal)
        assert hip.last_fwd_row_blocks() or not causal
        return [t.view(torch.int16) for t in (out.detach(), *(torch.autograd.grad(out, (qg, kg, vg), dout) if grad else ()))]

    _both(monkeypatch, run)


@pytest.mark.parametrize("D,chunks,rows,takes", [(64, 64, 2048, 1), (64, 65, 2048, 0), (96, 20, 2048, 0), (128, 20, 2048, 1), (256, 20, 2048, 1), (128, 20, 8, 0)])
def test_which_calls_choose_their_chunks_in_the_forward(D, chunks, rows, takes):
    f = hip.AttnFwdArgs()
    f.batch, f.total_q, f.total_k, f.heads, f.heads_k, f.head_dim = 2, 2 * rows, 128 * chunks, 8, 8, D
    f.max_seqlen_q, f.max_seqlen_k, f.max_cols, f.lg_block_n, f.is_causal, f.max_visits_per_row = rows, 64 * chunks, chunks, 64, 1, 24
    f.k_row_stride = f.v_row_stride = 8 * D
    assert hip.load_library().fmoba_attn_fwd_gates_rows(f) == takes
