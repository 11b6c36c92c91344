"""Uneven batches, whose grids hold the blocks that exist alone: every block has to be taken, once."""
import numpy as np
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip
from gpu_utils import assert_close
from test_gpu_item_order import _reference

pytestmark = pytest.mark.gpu


# Two sequences and as many as the look-up takes, one more; empty ones at the ends and between, all of one length but one; more than 64 blocks in the longest (two looks), at the edges of 64
# and 128; blocks of 64, 128 and 256 rows, 64 and 128 keys; one and two sets of waves, row blocks and columns, wide heads; heads of an XCD, of two, grouped; a bound longer than every sequence
@pytest.mark.parametrize("lens,H,Hk,D,chunk,topk,bound", [
    ([1300, 40], 8, 8, 64, 64, 4, 0), ([0, 700, 0, 64, 65, 1, 0], 16, 4, 128, 64, 3, 0), ([900] + [30 + i for i in range(31)], 8, 8, 64, 64, 3, 0),
    ([900] + [30 + i for i in range(32)], 8, 8, 64, 64, 3, 0), ([4097, 100, 5], 8, 8, 64, 64, 20, 0), ([4160, 64, 63], 8, 2, 64, 64, 3, 0), ([100, 3000, 129], 16, 16, 96, 128, 2, 0),
    ([100, 2600, 127, 300], 8, 8, 128, 128, 2, 0), ([1500, 256, 20, 257, 90], 16, 8, 256, 64, 8, 0), ([40, 2100, 200], 8, 8, 200, 64, 2, 0), ([500, 20, 30], 24, 8, 128, 64, 3, 5000),
    ([8200, 33, 40], 8, 1, 64, 64, 2, 0), ([60, 3000, 40, 20, 130], 8, 8, 128, 64, 2, 0), ([6500, 127, 40, 20], 16, 4, 128, 128, 2, 0)])
def test_every_block_once(lens, H, Hk, D, chunk, topk, bound):
    _every_block_once(lens, H, Hk, D, chunk, topk, bound, torch.bfloat16)


def _every_block_once(lens, H, Hk, D, chunk, topk, bound, dtype):
    """Result and gradients against the pattern's in fp32; returns whether the backward left dQ in partials."""
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + D)
    mk = lambda h: torch.randn((sum(lens), h, D), generator=g, device="cuda").to(dtype)
    q, k, v, dout = (x.requires_grad_(True) for x in (mk(H), mk(Hk), mk(Hk), mk(H)))
    cu = [0] + [int(x) for x in np.cumsum(lens)]
    cud, longest = torch.tensor(cu, dtype=torch.int32, device="cuda"), max(*lens, bound)
    form = []
    q.register_hook(lambda _: form.append(hip.last_bwd_partials()))  # (on the engine's thread, as the backward)
    out = flash_moba.flash_moba_varlen_func(q, k, v, cud, cud, longest, longest, chunk, topk, causal=True)
    got = (out.detach(), *torch.autograd.grad(out, (q, k, v), dout.detach()))
    pattern = flash_moba.flash_topk_varlen_func(q.detach(), k.detach(), cud, cud, longest, longest, topk, chunk, causal=True)
    # (bounds as for the order of the items: test_gpu_item_order.py)
    want = _reference(q.detach(), k.detach(), v.detach(), dout.detach(), cu, *pattern, chunk)
    for name, x, y, n in zip(("out", "dq", "dk", "dv"), got, want, (1, 1, H // Hk, H // Hk)):
        assert_close(name, x, y, 2e-2 * n, 1e-2)
    again = flash_moba.flash_moba_varlen_func(q.detach(), k.detach(), v.detach(), cud, cud, longest, longest, chunk, topk, causal=True)
    assert torch.equal(again, got[0])
    return form[0]


# dK/dV with partials, whose blocks are looked up where a plain grid has three times as many as there may be: blocks of 64 keys and of 128, empty sequences, a bound longer than every sequence
@pytest.mark.parametrize("lens,H,Hk,chunk,topk,bound", [
    ([5200, 100, 20, 40], 8, 8, 64, 1, 0), ([20, 0, 11000, 65], 8, 2, 64, 2, 0), ([6500, 127, 40, 20], 16, 4, 128, 2, 0), ([129, 7000, 0, 128], 8, 8, 128, 2, 9000)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_block_of_a_backward_with_partials_once(lens, H, Hk, chunk, topk, bound, dtype):
    keys = hip.fwd_key_block(chunk)  # (of a block of this pass too)
    assert len(lens) * -(-max(*lens, bound) // keys) >= 3 * (sum(lens) // keys + len(lens))
    assert _every_block_once(lens, H, Hk, 128, chunk, topk, bound, dtype) == 1


# later parts of prompts, by columns: keys and queries of other lengths, blocks by pairs (many keys) and by length
@pytest.mark.parametrize("lens_q,lens_k,H,Hk,D,chunk,topk", [
    ([300, 1, 0, 64], [20000, 700, 50, 3000], 16, 8, 64, 128, 4), ([200, 90, 33], [60000, 1000, 9000], 16, 8, 128, 128, 3), ([129, 70], [66, 5000], 8, 8, 128, 64, 2)])
def test_every_block_of_keys_once(lens_q, lens_k, H, Hk, D, chunk, topk):
    g = torch.Generator(device="cuda").manual_seed(sum(lens_k) + D)
    mk = lambda n, h: torch.randn((n, h, D), generator=g, device="cuda").to(torch.float16)
    q, k, v = mk(sum(lens_q), H), mk(sum(lens_k), Hk), mk(sum(lens_k), Hk)
    cq, ck = ([0] + [int(x) for x in np.cumsum(n)] for n in (lens_q, lens_k))
    dev = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    out = flash_moba.flash_moba_varlen_func(q, k, v, dev(cq), dev(ck), max(lens_q), max(lens_k), chunk, topk, causal=True)
    for b in range(len(lens_q)):  # alone: one sequence has no blocks that do not exist
        if lens_q[b] == 0:
            continue
        qs, ks = slice(cq[b], cq[b + 1]), slice(ck[b], ck[b + 1])
        one = flash_moba.flash_moba_varlen_func(q[qs], k[ks], v[ks], dev([0, lens_q[b]]), dev([0, lens_k[b]]), lens_q[b], lens_k[b], chunk, topk, causal=True)
        assert_close("out", out[qs], one.float().cpu(), 2e-3, 2e-3)  # fp16 results and partial rows, a rounding of 2^-11 each way
