"""Row-block forward of head dimensions above 128: edges of its tiles, its rule, its precision beside the column form's."""
import ctypes

import numpy as np
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip
from gpu_utils import assert_close
from gpu_utils import pattern_forward
from test_form_rules import fwd_args
from test_gpu_item_order import _reference


# 0.36 of the visible chunks with 128-key blocks (0.18 with 64-key ones), from one block of 128 rows per compute unit on
@pytest.mark.parametrize("lens,chunk,topk,heads,rows", [([16384], 128, 22, 4, 0), ([16384], 128, 23, 4, 1), ([16384], 64, 22, 4, 0), ([16384], 64, 23, 4, 1),
                                                        ([4096, 4096], 128, 8, 3, 0), ([4096, 4096], 128, 8, 4, 1)])
def test_wide_forward_lines(lens, chunk, topk, heads, rows):
    f = fwd_args(lens, chunk, topk, heads=heads, D=256)
    assert hip.load_library().fmoba_attn_fwd_uses_row_blocks(ctypes.byref(f)) == rows


# the density is that of the rows: most of them in the longest sequence of a batch, the last of their sequences in a part of a prompt
@pytest.mark.parametrize("lens_q,lens_k,chunk,topk,heads,rows", [
    ([637, 12295], None, 128, 13, 16, 0), ([6466, 6466], None, 128, 13, 16, 1), ([2789, 25592, 2556, 1271, 1642, 2226], None, 256, 3, 8, 0),
    ([1451, 156, 137], [11481, 479, 1317], 64, 7, 32, 0), ([1024, 1024], [4096, 4096], 128, 9, 32, 0), ([1024, 1024], [4096, 4096], 128, 11, 32, 1)])
def test_wide_forward_lines_of_uneven_calls(lens_q, lens_k, chunk, topk, heads, rows):
    lens_k = lens_k or lens_q
    f = fwd_args(lens_k, chunk, topk, heads=heads, D=256)
    f.total_q, f.max_seqlen_q = sum(lens_q), max(lens_q)
    assert hip.load_library().fmoba_attn_fwd_uses_row_blocks(ctypes.byref(f)) == rows


# keys or values further apart than the kernel's 32-bit offsets reach stay with the columns
@pytest.mark.parametrize("field", ["k_row_stride", "v_row_stride"])
def test_wide_forward_of_rows_far_apart(field):
    f = fwd_args([16384], 64, 32, heads=4, D=256)
    for stride, rows in ((1024, 1), ((1 << 24) - 8, 1), (1 << 24, 0), (1 << 26, 0)):
        setattr(f, field, stride)
        assert hip.load_library().fmoba_attn_fwd_uses_row_blocks(ctypes.byref(f)) == rows


def _inputs(lens, H, Hk, D, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn((sum(lens), h, D), generator=g, device="cuda").to(dtype) for h in (H, Hk, Hk))
    cu = [0] + [int(x) for x in np.cumsum(lens)]
    return q, k, v, cu, torch.tensor(cu, dtype=torch.int32, device="cuda")


def _forward(q, k, v, cu, lens, pattern, chunk, mode):
    out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, *pattern, cu, cu, None, None, None, max(lens), max(lens), 0.0, q.shape[2] ** -0.5, False, True, 0.0,
                                         False, 128, chunk, None, _fwd_mode=mode)
    return out, lse


# walks of one step and of two, rows and keys at the edges of 32, 64 and 128, a last chunk cut short, feature pieces that do not exist,
# key heads that are shared, more than one word of selection bits
@pytest.mark.gpu
@pytest.mark.parametrize("lens,H,Hk,D,chunk,topk", [
    ([1, 31, 32, 33, 0, 63, 64, 65], 2, 2, 256, 64, 2), ([127, 128, 129, 193, 257], 4, 1, 136, 64, 3), ([385, 700], 2, 1, 192, 256, 2),
    ([2300], 2, 2, 256, 64, 20), ([513, 1100], 2, 2, 248, 128, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_wide_row_blocks(lens, H, Hk, D, chunk, topk, dtype):
    q, k, v, cu, cud = _inputs(lens, H, Hk, D, dtype, sum(lens) + D)
    pattern = flash_moba.flash_topk_varlen_func(q, k, cud, cud, max(lens), max(lens), topk, chunk, causal=True)
    out, lse = _forward(q, k, v, cud, lens, pattern, chunk, 2)
    # (the bound of the other attention tests)
    assert_close("out", out, _reference(q, k, v, torch.zeros_like(q), cu, *pattern, chunk)[0], 2e-2, 1e-2)
    # the column form's sums of the same scores are fp32 too: the two differ by the order of some 2500 of them
    assert (lse - _forward(q, k, v, cud, lens, pattern, chunk, 1)[1]).abs().nan_to_num(0.0).max() <= 1e-4


# equal scores: every probability is a power of two, a row the mean of its values, rounded once
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_wide_row_blocks_round_once(dtype):
    L, D, chunk = 900, 256, 64
    q, k, v, _, cud = _inputs([L], 2, 2, D, dtype, 3)
    q, v = torch.zeros_like(q), v.abs() + 0.5
    pattern = flash_moba.flash_topk_varlen_func(q, k, cud, cud, L, L, 15, chunk, causal=True)
    out, _ = _forward(q, k, v, cud, [L], pattern, chunk, 2)
    exact = v.double().cumsum(0) / torch.arange(1, L + 1, device="cuda", dtype=torch.float64)[:, None, None]
    half_ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) * (1 + 2 ** -6)  # and the 32-bit sums under it
    assert ((out.double() - exact).abs() <= half_ulp * exact).all()


# scores that grow by up to 2^10 from block to block and fall again, scores of -inf, and rows whose unselected chunks hold infinite ones
@pytest.mark.gpu
def test_wide_row_blocks_extreme_scores():
    L, D, chunk = 640, 256, 64
    q, k, v, cu, cud = _inputs([L], 1, 1, D, torch.bfloat16, 5)
    size = torch.tensor([1.0, 30.0, 0.01, 120.0, 5.0, 60.0, 0.5, 90.0, 2.0, 1.0], device="cuda").repeat_interleave(chunk)
    k = (k.float() * size[:, None, None]).to(k.dtype)
    pattern = flash_moba.flash_topk_varlen_func(q, k, cud, cud, L, L, 10, chunk, causal=True)
    rows, _ = _forward(q, k, v, cud, [L], pattern, chunk, 2)
    want = _reference(q, k, v, torch.zeros_like(q), cu, *pattern, chunk)[0]
    assert_close("out", rows, want, 2e-2, 1e-2)
    q = q.abs() + 0.1
    k[3 * chunk:4 * chunk] = float("-inf")  # selected by rows that have no more than their own chunk and this one alone
    pattern = flash_moba.flash_topk_varlen_func(q, k, cud, cud, L, L, 3, chunk, causal=True)
    rows, rows_lse = _forward(q, k, v, cud, [L], pattern, chunk, 2)
    cols, cols_lse = _forward(q, k, v, cud, [L], pattern, chunk, 1)
    assert torch.equal(rows.isnan(), cols.isnan()) and torch.equal(rows_lse.isinf(), cols_lse.isinf())
    assert_close("out", rows.nan_to_num(0.0), cols.nan_to_num(0.0), 2e-2, 1e-2)
    k[3 * chunk:4 * chunk] = float("inf")
    pattern = [t.clone() for t in pattern]  # rows of a pattern that leaves those keys out
    pattern[1][0, 0, 3] = 0
    rows, _ = _forward(q, k, v, cud, [L], pattern, chunk, 2)
    cols, _ = _forward(q, k, v, cud, [L], pattern, chunk, 1)
    assert_close("out", rows, cols, 2e-2, 1e-2)


# The largest probability of a block is a power of two, which 16 bits hold exactly, as in the column form, whose blocks are as long or
# longer: the error against 32-bit attention is no larger (1 % for the sample)
@pytest.mark.gpu
@pytest.mark.parametrize("chunk,topk", [(64, 8), (128, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_wide_row_blocks_are_as_precise_as_columns(chunk, topk, dtype):
    lens = [2048]
    q, k, v, cu, cud = _inputs(lens, 4, 4, 256, dtype, 7)
    pattern = flash_moba.flash_topk_varlen_func(q, k, cud, cud, 2048, 2048, topk, chunk, causal=True)
    want = _reference(q, k, v, torch.zeros_like(q), cu, *pattern, chunk)[0]
    err = [float((_forward(q, k, v, cud, lens, pattern, chunk, m)[0].float() - want).norm()) for m in (2, 1)]
    assert err[0] <= err[1] * 1.01


# rows of q and dout that 32-bit byte offsets do not reach (2^22 elements apart): the bits of the packed tensors
@pytest.mark.gpu
@pytest.mark.parametrize("D,chunk", [(256, 64), (192, 128)])
def test_wide_backward_with_rows_far_apart(D, chunk):
    lens = [150, 70]
    q, k, v, _, cu = _inputs(lens, 2, 2, D, torch.bfloat16, D)
    dout = _inputs(lens, 2, 2, D, torch.bfloat16, D + 1)[0]
    pattern = flash_moba.flash_topk_varlen_func(q, k, cu, cu, 150, 150, 2, chunk, causal=True)
    out, lse = _forward(q, k, v, cu, lens, pattern, chunk, 0)
    far = lambda t: torch.empty((220, 1 << 22), dtype=t.dtype, device="cuda")[:, :2 * D].view(220, 2, D).copy_(t)
    grads = lambda q, dout: hip.moba_varlen_bwd(dout, q, k, v, out, lse, None, None, None, *pattern, cu, cu, None, 150, 150, 0.0, D ** -0.5, False, True, 0.0,
                                                False, 128, chunk, None)[:3]
    for near, apart in zip(grads(q, dout), grads(far(q), far(dout))):
        assert torch.equal(near, apart)


# infinities and NaN in Q and K: the same elements of out and lse are NaN and infinite as in the column form, the others agree
@pytest.mark.gpu
@pytest.mark.parametrize("which,at,value", [("q", 300, float("nan")), ("q", 300, float("inf")), ("k", 200, float("nan")), ("k", 200, float("inf")),
                                            ("k", 200, float("-inf")), ("k", slice(192, 256), float("nan"))])
@pytest.mark.parametrize("D", [256, 136])
def test_wide_row_blocks_non_finite_scores(which, at, value, D):
    L, chunk = 700, 64
    q, k, v, cu, cud = _inputs([L], 2, 1, D, torch.bfloat16, 11)
    pattern = flash_moba.flash_topk_varlen_func(q, k, cud, cud, L, L, 4, chunk, causal=True)
    {"q": q, "k": k}[which][at, 0] = value
    _assert_same_places(_forward(q, k, v, cud, [L], pattern, chunk, 2), _forward(q, k, v, cud, [L], pattern, chunk, 1))


def _assert_same_places(got, want):
    for x, y in zip(got, want):
        assert torch.equal(x.isnan(), y.isnan()) and torch.equal(x.isposinf(), y.isposinf()) and torch.equal(x.isneginf(), y.isneginf())
        assert_close("row blocks", x.nan_to_num(0.0, 0.0, 0.0), y.nan_to_num(0.0, 0.0, 0.0), 2e-2, 1e-2)  # (the bounds of the other attention tests)


# infinities and NaN in V: they reach the rows that selected their chunk, as in the column form, and no bit of the others; a head apart, pieces at the end of
# the features, the last key of a sequence, a row block whose walk is one step
@pytest.mark.gpu
@pytest.mark.parametrize("at,feature,value", [(70, 3, float("inf")), (255, 100, float("nan")), (400, -1, float("-inf")), (699, 0, float("inf")), (720, 8, float("nan")),
                                              (1, slice(None), float("inf"))])
@pytest.mark.parametrize("D", [256, 136])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_wide_row_blocks_non_finite_values(at, feature, value, D, dtype):
    lens, chunk = [700, 40, 300], 64
    q, k, v, cu, cud = _inputs(lens, 4, 2, D, dtype, 12)
    pattern = flash_moba.flash_topk_varlen_func(q, k, cud, cud, max(lens), max(lens), 4, chunk, causal=True)
    plain, _ = _forward(q, k, v, cud, lens, pattern, chunk, 2)
    v[at, 1, feature] = value
    rows, cols = (_forward(q, k, v, cud, lens, pattern, chunk, m) for m in (2, 1))
    _assert_same_places(rows, cols)
    b = 0 if at < 700 else 1
    c = (at - cu[b]) // chunk
    hit = torch.zeros(q.shape[:2], dtype=torch.bool, device="cuda")
    for h in (2, 3):
        lo, n = int(pattern[0][b, h, c]), int(pattern[1][b, h, c])
        hit[cu[b] + pattern[2][lo:lo + n].long(), h] = True
    assert hit.any() and not hit.all() and torch.equal(rows[0][~hit], plain[~hit])


# later parts of prompts, more queries than keys (the first rows see nothing: out 0, lse +inf, whole blocks of them), no causal limit; a last chunk cut short
@pytest.mark.gpu
@pytest.mark.parametrize("lens_q,lens_k", [([200, 1, 130], [1000, 65, 131]), ([700, 300, 40], [150, 300, 1]), ([129, 257], [2100, 64])])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D,chunk", [(256, 64), (192, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_wide_row_blocks_of_unequal_lengths(lens_q, lens_k, causal, D, chunk, dtype):
    g = torch.Generator(device="cuda").manual_seed(sum(lens_k) + D)
    q, k, v = (torch.randn((sum(n), h, D), generator=g, device="cuda").to(dtype) for n, h in ((lens_q, 4), (lens_k, 2), (lens_k, 2)))
    cu_q, cu_k = ([0] + [int(x) for x in np.cumsum(lens)] for lens in (lens_q, lens_k))
    where = (*(torch.tensor(x, dtype=torch.int32, device="cuda") for x in (cu_q, cu_k)), max(lens_q), max(lens_k))
    pattern = flash_moba.flash_topk_varlen_func(q, k, *where, 6, chunk, causal=causal)
    out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, *pattern, *where[:2], None, None, None, *where[2:], 0.0, D ** -0.5, False, causal, 0.0, False, 128, chunk, None,
                                         _fwd_mode=2)
    assert hip.last_fwd_row_blocks()
    want, want_lse = pattern_forward(q, k, v, cu_q, cu_k, *pattern, chunk, causal)
    assert_close("out", out, want, 2e-2, 1e-2)  # (the bound of the other attention tests)
    assert torch.equal(lse.isinf(), want_lse.isinf()) and torch.equal(out[(want_lse.T == float("inf"))], torch.zeros_like(out[(want_lse.T == float("inf"))]))
    # (256 products and 1100 probabilities per sum in 32 bits, in another order; scores of up to 2^3 in magnitude)
    assert (lse - want_lse).nan_to_num(0.0).abs().max() <= 1e-3
