"""Which form a call runs (host rules of the library), at the lines the rules draw."""
import ctypes

import pytest

from flash_moba import flash_moba_hip as H


def fwd_args(lens, chunk, topk, heads=4, D=128, causal=1):
    f = H.AttnFwdArgs()
    f.total_q = f.total_k = sum(lens)
    f.heads = f.heads_k = heads
    f.head_dim, f.batch, f.lg_block_n, f.is_causal = D, len(lens), chunk, causal
    f.max_seqlen_q = f.max_seqlen_k = max(lens)
    f.max_cols = -(-max(lens) // chunk)
    f.max_visits_per_row = topk * (chunk // H.fwd_key_block(chunk))
    return f


# a row whose visits were added up in fp32 is not handed to 16-bit partial rows for speed: 128-key blocks stay on row blocks
# from 10/27 of the visible chunks on, 64-key blocks from 10/50
@pytest.mark.parametrize("chunk,topk,rows", [(128, 23, 0), (128, 24, 1), (128, 26, 1), (256, 11, 0), (256, 12, 1), (64, 25, 0), (64, 26, 1)])
def test_forward_lines(chunk, topk, rows):
    f = fwd_args([16384], chunk, topk)
    assert H.load_library().fmoba_attn_fwd_uses_row_blocks(ctypes.byref(f)) == rows


# the same for dQ: fp32 sums over dS tiles from a tenth of the visible chunks on with 64-key blocks and with heads up to 64,
# from 0.37 on with 128-key blocks
@pytest.mark.parametrize("D,chunk,topk,partials", [(128, 64, 12, 1), (128, 64, 13, 0), (128, 64, 18, 0), (64, 64, 12, 1), (64, 64, 13, 0), (64, 64, 28, 0),
                                                   (64, 128, 6, 1), (64, 128, 7, 0), (96, 128, 23, 1), (128, 128, 23, 1), (128, 128, 24, 0), (256, 64, 1, 0)])
def test_dq_lines(D, chunk, topk, partials):
    a = H.AttnBwdArgs()
    a.total_q = a.total_k = a.max_seqlen_q = a.max_seqlen_k = 16384
    a.heads = a.heads_k = 4
    a.head_dim, a.batch, a.lg_block_n, a.is_causal = D, 1, chunk, 1
    a.max_visits_per_row = topk * (chunk // 64)
    assert H.load_library().fmoba_attn_bwd_uses_partials(ctypes.byref(a)) == partials


# above head dimension 128 the partial results of a row are bounded by the key blocks of a sequence, whatever top-k times the chunk
# is, and calls whose rows still have more of them than the combine can order go to row blocks
def test_wide_heads_partial_results_are_bounded_by_the_sequence():
    lib = H.load_library()
    f = fwd_args([512], 4096, 64, heads=2, D=256)
    assert lib.fmoba_attn_fwd_uses_row_blocks(ctypes.byref(f)) == 0
    assert lib.fmoba_attn_fwd_workspace_bytes(ctypes.byref(f)) < 512 * 2 * 4 * (4 * 256 + 16) + 8192
    f = fwd_args([512], 64 * 129, 64, heads=2, D=256)
    f.total_k = f.max_seqlen_k = 200000
    f.max_cols = 25
    assert lib.fmoba_attn_fwd_uses_row_blocks(ctypes.byref(f)) == 1
    f.total_k = f.max_seqlen_k = 160000
    f.max_cols = 20
    assert lib.fmoba_attn_fwd_uses_row_blocks(ctypes.byref(f)) == 0


# visits of a pattern: in LDS for calls worth at least twelve heads of the longest sequence (more of them where a sequence has few), by atomics where one
# workgroup would read most of the call's lists
@pytest.mark.parametrize("lens,heads,lds", [([262144], 8, 0), ([262144], 11, 0), ([262144], 12, 1), ([200000] + [2048] * 7, 1, 0), ([150000] + [2000] * 7, 4, 0),
                                            ([20000] * 63, 1, 0), ([20000] * 64, 1, 1), ([20000] * 15, 2, 0), ([20000] * 16, 2, 1), ([20000] * 4, 4, 1),
                                            ([1024], 8, 1), ([1024], 7, 0), ([2304], 8, 0)])
def test_visits_in_lds(lens, heads, lds):
    assert H.load_library().fmoba_csc_row_visits_in_lds(ctypes.byref(fwd_args(lens, 128, 16, heads=heads))) == lds


# four sets of waves share a walk of 16 steps and more in calls of few row blocks of narrow heads: not the short ones, which they only make longer
@pytest.mark.parametrize("lens,heads,D,sets", [([64] * 2, 4, 64, 2), ([896] * 2, 4, 64, 2), ([1023], 8, 64, 2), ([1024], 8, 64, 4), ([1024] * 2, 8, 64, 2), ([2048], 8, 64, 4),
                                               ([2112], 8, 64, 2), ([1024], 8, 72, 2), ([8192], 8, 32, 2), ([8832], 8, 64, 1), ([4480], 8, 128, 2), ([4736], 8, 128, 1)])
def test_sets_of_a_walk(lens, heads, D, sets):
    assert H.load_library().fmoba_attn_fwd_row_sets(ctypes.byref(fwd_args(lens, 64, 16, heads=heads, D=D))) == sets


# the form that chooses its rows' chunks itself reads no selection bits: a struct that still holds some from another call is of the form as well
@pytest.mark.parametrize("lens,D,gated", [([2048], 64, 1), ([4096], 128, 1), ([2048], 256, 1), ([2048], 96, 0), ([4160], 64, 0)])
def test_gated_row_blocks_whatever_selection_bits(lens, D, gated):
    f = fwd_args(lens, 64, 20, heads=16, D=D)
    for f.selection_bits in (None, 4096):
        assert H.load_library().fmoba_attn_fwd_gates_rows(ctypes.byref(f)) == gated
