"""dK / dV of query heads that share keys, added up inside the kernel: any number of heads of a group."""
import numpy as np
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip
from gpu_utils import assert_close

pytestmark = pytest.mark.gpu


class _Library:
    """the loaded library, but for the number of heads it asks for"""

    def __init__(self, lib, heads):
        self._lib, self.fmoba_attn_bwd_dkv_heads = lib, lambda args: heads

    def __getattr__(self, name):
        return getattr(self._lib, name)


# lists of a group that end in the middle of a round, have no rows at all (non-causal, few rows), start past a block's first
# rows (chunks of three blocks); keys past the last query; a group of one, of some, of all heads, of a whole wave
@pytest.mark.parametrize("lens_q,lens_k,chunk,topk,causal", [
    ([700, 65, 1], [700, 65, 1], 64, 3, True), ([1000], [1500], 192, 2, True), ([3, 0, 130], [900, 64, 257], 128, 1, False)])
@pytest.mark.parametrize("H,Hk,counts", [(8, 1, (1, 2, 4)), (6, 2, (2,)), (64, 1, (1, 2))])
@pytest.mark.parametrize("D,dq_mode", [(64, 1), (64, 2), (40, 2), (128, 1), (96, 1)])
def test_groups_add_up(lens_q, lens_k, chunk, topk, causal, H, Hk, counts, D, dq_mode, monkeypatch):
    g = torch.Generator().manual_seed(H + D + chunk)
    mk = lambda n, h: torch.randn((n, h, D), generator=g).to(torch.bfloat16).cuda()
    cu = lambda lens: torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32).cuda()
    q, k, v, dout, cuq, cuk = mk(sum(lens_q), H), mk(sum(lens_k), Hk), mk(sum(lens_k), Hk), mk(sum(lens_q), H), cu(lens_q), cu(lens_k)
    mq, mk_ = max(lens_q), max(lens_k)
    co, cn, ind = flash_moba.flash_topk_varlen_func(q, k, cuq, cuk, mq, mk_, topk, chunk, causal=causal)
    out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, co, cn, ind, cuq, cuk, None, None, None, mq, mk_, 0.0, D ** -0.5,
                                         False, causal, 0.0, False, 128, chunk, None)
    lib = hip.load_library()

    def grads(heads, k, v):
        monkeypatch.setattr(hip, "load_library", lambda: _Library(lib, heads))
        return hip.moba_varlen_bwd(dout, q, k, v, out, lse, None, None, None, co, cn, ind, cuq, cuk, None, mq, mk_, 0.0, D ** -0.5,
                                   False, causal, 0.0, False, 128, chunk, _dq_mode=dq_mode)[:3]

    dq, dk, dv = grads(H, k.repeat_interleave(H // Hk, 1), v.repeat_interleave(H // Hk, 1))  # a head of keys per query head
    dk, dv = (t.float().view(-1, Hk, H // Hk, D) for t in (dk, dv))
    for n in counts:
        dq2, dk2, dv2 = grads(n, k, v)
        if dq_mode == 1:
            assert torch.equal(dq, dq2)
        else:  # which visit got which slot does not matter: a row's visits are ordered before they are added
            assert_close("dq", dq2, dq.float().cpu(), 2e-2, 1e-2)
        for name, got, ref in (("dk", dk2, dk), ("dv", dv2, dv)):  # (every term of the sum was rounded to 16 bits, and so are partial sums)
            worst = (got.float() - ref.sum(2)).abs() - 2.0 ** -7 * ref.abs().sum(2)
            assert worst.max().item() < 1e-3, f"{name}: {worst.max().item()}"


# rows of q and dout that 32-bit byte offsets do not reach (2^22 elements apart), in a walk over several heads: the bits of the packed tensors
@pytest.mark.parametrize("D,dq_mode", [(128, 1), (96, 1), (64, 1), (64, 2)])
def test_groups_of_rows_far_apart(D, dq_mode, monkeypatch):
    L, H, chunk = 150, 4, 64
    g = torch.Generator().manual_seed(D)
    mk = lambda h: torch.randn((L, h, D), generator=g).to(torch.bfloat16).cuda()
    q, k, v, dout, cu = mk(H), mk(1), mk(1), mk(H), torch.tensor([0, L], dtype=torch.int32).cuda()
    pattern = flash_moba.flash_topk_varlen_func(q, k, cu, cu, L, L, 2, chunk, causal=True)
    out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, *pattern, cu, cu, None, None, None, L, L, 0.0, D ** -0.5, False, True, 0.0, False, 128, chunk, None)
    lib = hip.load_library()
    monkeypatch.setattr(hip, "load_library", lambda: _Library(lib, 1))

    def far(t):
        view = torch.empty((L, 1 << 22), dtype=t.dtype, device="cuda")[:, :H * D].view(L, H, D)
        return view.copy_(t)

    grads = lambda q, dout: hip.moba_varlen_bwd(dout, q, k, v, out, lse, None, None, None, *pattern, cu, cu, None, L, L, 0.0, D ** -0.5,
                                                False, True, 0.0, False, 128, chunk, _dq_mode=dq_mode)[:3]
    for near, apart in zip(grads(q, dout), grads(far(q), far(dout))):
        assert torch.equal(near, apart)
