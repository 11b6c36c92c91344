"""Lists with ranks (native host path) against plain lists whose rows hand out places from counters (path through the ops): same bits."""
import numpy as np
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip
from test_gpu_host_path import _both

pytestmark = pytest.mark.gpu


# Columns with partial rows of dQ: one key block per chunk, two and four, two in the backward alone (heads of 64), the last chunk cut
# short, more than eight words of selection per row, more heads in a group than a workgroup takes.  Columns with dS tiles: three
# blocks per chunk, wide heads.  Row blocks with partial rows of dQ.  Sequences of one row and none; queries that are the last rows of
# their sequence; the plain rule
@pytest.mark.parametrize("lens_q,lens_k,H,Hk,D,chunk,topk,causal,rows,partials", [
    ([4100], [4100], 2, 2, 128, 128, 4, True, 0, 1), ([12007, 1, 0, 300], [12007, 1, 0, 300], 2, 1, 72, 256, 2, True, 0, 1),
    ([9000], [9000], 1, 1, 128, 512, 2, True, 0, 1), ([8001], [8001], 2, 2, 64, 128, 2, True, 0, 1), ([20000], [20000], 2, 2, 32, 64, 5, True, 0, 1),
    ([5, 900], [7000, 9100], 4, 1, 128, 128, 4, True, 0, 1), ([5000, 77], [5000, 77], 2, 2, 128, 256, 3, False, 0, 1),
    ([2000], [2000], 132, 1, 64, 64, 1, True, 0, 1), ([6000], [6000], 2, 2, 96, 192, 2, True, 0, 0), ([3000, 200], [3000, 200], 2, 2, 256, 128, 4, True, 0, 0),
    ([5, 3], [7000, 9100], 4, 1, 128, 128, 4, True, 1, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_ranked_lists_give_the_bits_of_counted_places(monkeypatch, lens_q, lens_k, H, Hk, D, chunk, topk, causal, rows, partials, dtype):
    g = torch.Generator(device="cuda").manual_seed(sum(lens_q) + D)
    mk = lambda n, h: torch.randn((n, h, D), generator=g, device="cuda").to(dtype)
    q, k, v, dout = mk(sum(lens_q), H), mk(sum(lens_k), Hk), mk(sum(lens_k), Hk), mk(sum(lens_q), H)
    q[-3, 0] = float("inf")  # rows whose scores are infinite or undefined
    q[-7, 0] = float("nan")
    cq, ck = (torch.tensor([0] + list(np.cumsum(x)), dtype=torch.int32, device="cuda") for x in (lens_q, lens_k))

    def run():
        qg, kg, vg = (t.clone().requires_grad_(True) for t in (q, k, v))
        seen = []
        qg.register_hook(lambda _: seen.append(hip.last_bwd_partials()))  # (on the engine's thread, as the backward)
        out = flash_moba.flash_moba_varlen_func(qg, kg, vg, cq, ck, max(lens_q), max(lens_k), chunk, topk, causal=causal)
        assert hip.last_fwd_row_blocks() == rows
        out.backward(dout)
        assert seen == [partials]
        return [t.view(torch.int16) for t in (out.detach(), qg.grad, kg.grad, vg.grad)]

    _both(monkeypatch, run)


# A buffer longer than its batch, at both ends: rows that belong to no sequence come out as with plain lists, whatever the memory of the
# call held before (NaN here).  One word of selection per row and several, partial rows in 16 bits and in fp32, row blocks with
# partial rows of dQ; more such rows than a block of the scan has threads
@pytest.mark.parametrize("lens_q,lens_k,before,after,H,D,chunk,topk,rows,partials", [
    ([4100, 300], [4100, 300], 3, 700, 2, 128, 128, 2, 0, 1), ([9000], [9000], 300, 1, 2, 64, 128, 2, 0, 1), ([2100], [2100], 0, 3000, 2, 256, 128, 4, 0, 0),
    ([5, 3], [7000, 9100], 2, 9, 2, 128, 128, 4, 1, 1)])
def test_rows_of_no_sequence_are_zero(monkeypatch, lens_q, lens_k, before, after, H, D, chunk, topk, rows, partials):
    g = torch.Generator(device="cuda").manual_seed(D)
    nq = sum(lens_q) + before + after
    mk = lambda n: torch.randn((n, H, D), generator=g, device="cuda").to(torch.bfloat16)
    q, k, v, dout = mk(nq), mk(sum(lens_k)), mk(sum(lens_k)), mk(nq)
    cq = before + torch.tensor([0] + list(np.cumsum(lens_q)), dtype=torch.int32, device="cuda")
    ck = torch.tensor([0] + list(np.cumsum(lens_k)), dtype=torch.int32, device="cuda")

    def run():
        qg, kg, vg = (t.clone().requires_grad_(True) for t in (q, k, v))
        seen = []
        qg.register_hook(lambda _: seen.append(hip.last_bwd_partials()))
        nan = [torch.full((n >> 2,), 0x7fc07fc0, dtype=torch.int32, device="cuda") for n in [1 << 19] * 32 + [1 << 24] * 16 + [1 << 28]]
        del nan
        out = flash_moba.flash_moba_varlen_func(qg, kg, vg, cq, ck, max(lens_q), max(lens_k), chunk, topk, causal=True)
        assert hip.last_fwd_row_blocks() == rows
        nan = [torch.full((n >> 2,), 0x7fc07fc0, dtype=torch.int32, device="cuda") for n in [1 << 19] * 32 + [1 << 24] * 16 + [1 << 28]]
        del nan
        out.backward(dout)
        assert seen == [partials]
        own = slice(before, nq - after)
        for t in ([] if rows else [out.detach()]) + ([qg.grad] if partials else []):  # (the other forms leave such rows alone)
            assert not torch.cat([t[:before], t[nq - after:]]).any()
        return [t.view(torch.int16) for t in (out.detach()[own], qg.grad[own], kg.grad, vg.grad)]

    _both(monkeypatch, run)


def test_ranked_lists_hold_the_rows_of_plain_ones():
    """Row | rank << 24, as the entry point documents it, and the visits of every row."""
    import ctypes
    L, H, D, chunk, topk = 3000, 2, 64, 64, 5
    g = torch.Generator(device="cuda").manual_seed(0)
    q, k = (torch.randn((L, H, D), generator=g, device="cuda").to(torch.bfloat16) for _ in range(2))
    cu = torch.tensor([0, L], dtype=torch.int32, device="cuda")
    co, cn, plain = flash_moba.flash_topk_varlen_func(q, k, cu, cu, L, L, topk, chunk, causal=True)
    lib, C = hip.load_library(), -(-L // chunk)
    km, cuk = torch.empty((C + 1, H, D), dtype=q.dtype, device="cuda"), torch.empty(2, dtype=torch.int32, device="cuda")
    co2, cn2, ranked = torch.empty_like(co), torch.empty_like(cn), torch.empty_like(plain)
    visits, prefix = torch.empty((H, L), dtype=torch.int32, device="cuda"), torch.empty(H * -(-C // 32) * L, dtype=torch.uint8, device="cuda")
    nws = lib.fmoba_fused_topk_workspace_bytes(1, L, H, L, L, chunk)
    ws = torch.empty(nws, dtype=torch.uint8, device="cuda")
    m = hip.MeanPoolArgs(k.data_ptr(), km.data_ptr(), cu.data_ptr(), cuk.data_ptr(), 1, C, H, D, chunk, 1, H * D, D, H * D, D)
    a = hip.FusedTopkArgs(q.data_ptr(), km.data_ptr(), cu.data_ptr(), cu.data_ptr(), cuk.data_ptr(), co2.data_ptr(), cn2.data_ptr(), ranked.data_ptr(), None, None,
                          ws.data_ptr(), nws, 1, L, H, H, D, L, L, topk, chunk, 1, 1, H * D, D, H * D, D)
    r = hip.CscRanks(visits.data_ptr(), prefix.data_ptr())
    assert lib.fmoba_pool_and_gate_ranked(ctypes.byref(m), ctypes.byref(a), ctypes.byref(r), None) == 0, lib.fmoba_last_error()
    torch.cuda.synchronize()
    assert torch.equal(co, co2) and torch.equal(cn, cn2) and torch.equal(ranked & 0xffffff, plain)
    off, nnz, ranked = co.cpu().numpy()[0], cn.cpu().numpy()[0], ranked.cpu().numpy()
    for h in range(H):
        seen = np.zeros(L, dtype=np.int64)
        for c in range(C):
            e = ranked[off[h, c]:off[h, c] + nnz[h, c]]
            assert (e >> 24 == seen[e & 0xffffff]).all()
            seen[e & 0xffffff] += 1
        got = visits[h].cpu().numpy()
        assert (got & 0xffff == seen).all() and (got >> 16 == seen).all()


@pytest.mark.parametrize("lens,H,Hk,D,chunk,topk,rows,partials", [([4100, 3000], 4, 2, 128, 128, 3, 0, 1), ([9000], 2, 2, 64, 64, 5, 0, 1), ([2100], 2, 1, 256, 128, 4, 0, 0), ([700], 2, 2, 128, 64, 6, 1, 0)])
def test_attention_over_ranked_lists_by_hand(lens, H, Hk, D, chunk, topk, rows, partials):
    """pool_and_gate_ranked, then moba_varlen_fwd / _bwd with the visits: the bits of plain lists."""
    g = torch.Generator(device="cuda").manual_seed(sum(lens))
    mk = lambda h: torch.randn((sum(lens), h, D), generator=g, device="cuda").to(torch.bfloat16)
    q, k, v, dout = mk(H), mk(Hk), mk(Hk), mk(H)
    cu, n, scale = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32, device="cuda"), max(lens), D ** -0.5
    plain = list(flash_moba.flash_topk_varlen_func(q, k, cu, cu, n, n, topk, chunk, causal=True))
    *ranked, selection, visits = hip.pool_and_gate_ranked(q, k, cu, cu, n, n, topk, chunk, True)
    kb = hip.fwd_key_block(chunk)
    bound = topk * (chunk // kb)
    res = []
    for lists, kw in ((plain, {}), (ranked, {"_visits": visits})):
        sel = {"_selection": selection} if rows else {}  # (row blocks over ranked lists read the selection words)
        out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, *lists, cu, cu, None, None, None, n, n, 0.0, scale, False, True, 0.0, False, 128, chunk, None,
                                             _max_visits=bound, **sel, **kw)
        assert hip.last_fwd_row_blocks() == rows
        grads = hip.moba_varlen_bwd(dout, q, k, v, out, lse, None, None, None, *lists, cu, cu, None, n, n, 0.0, scale, False, True, 0.0, False, 128, chunk, None,
                                    _max_visits=bound * (kb // 64), **kw)
        assert hip.last_bwd_partials() == partials
        res.append([t.view(torch.int16) for t in (out, *grads[:3])])
    for name, a, b in zip(("out", "dq", "dk", "dv"), *res):
        assert torch.equal(a, b), name
    with pytest.raises(RuntimeError, match="bound"):
        hip.moba_varlen_fwd(q, k, v, None, *ranked, cu, cu, None, None, None, n, n, 0.0, scale, False, True, 0.0, False, 128, chunk, None, _visits=visits)
