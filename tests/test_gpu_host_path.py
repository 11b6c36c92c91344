"""The native eager host path against the path through the custom ops, which stays for traced calls: same bits."""
import numpy as np
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip

pytestmark = pytest.mark.gpu


class _NoHost:
    """A host module that takes no call."""

    def __getattr__(self, name):
        return lambda *a: None


def _both(monkeypatch, fn):
    got = fn()
    with monkeypatch.context() as m:
        m.setattr(hip, "host_module", lambda: _NoHost())
        want = fn()
    for x, y in zip(got, want):
        assert x.shape == y.shape and x.dtype == y.dtype and torch.equal(x, y)
    return got


# one row, uneven lengths with empty sequences, more sequences than a wave has lanes, more than the pooling counts itself
@pytest.mark.parametrize("lens_q,lens_k,H,Hk,D,chunk,topk", [
    ([1], [1], 1, 1, 8, 64, 1), ([300, 0, 77], [300, 0, 77], 4, 2, 64, 64, 3), ([5, 900], [700, 2000], 4, 1, 128, 128, 4),
    ([7] * 70, [7] * 70, 2, 2, 72, 64, 2), ([2] * 1030, [3] * 1030, 1, 1, 64, 64, 2), ([600], [600], 2, 2, 256, 64, 3),
    ([2500], [2500], 4, 4, 128, 64, 2)])
@pytest.mark.parametrize("grad", [False, True])
def test_native_host_path_gives_the_bits_of_the_op_path(monkeypatch, lens_q, lens_k, H, Hk, D, chunk, topk, grad):
    g = torch.Generator(device="cuda").manual_seed(sum(lens_q) + D)
    mk = lambda n, h: torch.randn((n, h, D), generator=g, device="cuda").to(torch.bfloat16)
    q, k, v, dout = mk(sum(lens_q), H), mk(sum(lens_k), Hk), mk(sum(lens_k), Hk), mk(sum(lens_q), H)
    cu = lambda lens: torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32, device="cuda")
    cq, ck = cu(lens_q), cu(lens_k)
    where = (cq, ck, max(lens_q), max(lens_k))

    def fused():
        qg, kg, vg = (t.clone().requires_grad_(grad) for t in (q, k, v))
        out = flash_moba.flash_moba_varlen_func(qg, kg, vg, *where, chunk, topk, causal=True)
        return (out.detach(),) + (torch.autograd.grad(out, (qg, kg, vg), dout) if grad else ())

    def two_step():
        qg, kg, vg = (t.clone().requires_grad_(grad) for t in (q, k, v))
        pattern = flash_moba.flash_topk_varlen_func(q, k, *where, topk, chunk, causal=True)
        out = flash_moba.flash_moba_attn_varlen_func(qg, kg, vg, *where, *pattern, lg_block_m=128, lg_block_n=chunk, causal=True)
        return (out.detach(), *pattern) + (torch.autograd.grad(out, (qg, kg, vg), dout) if grad else ())

    one = _both(monkeypatch, fused)
    two = _both(monkeypatch, two_step)
    assert torch.equal(one[0], two[0])


def test_gradients_have_no_gradients():
    x = torch.randn((200, 2, 64), device="cuda").to(torch.bfloat16).requires_grad_(True)
    cu = torch.tensor([0, 200], dtype=torch.int32, device="cuda")
    out = flash_moba.flash_moba_varlen_func(x, x, x, cu, cu, 200, 200, 64, 2)
    (dx,) = torch.autograd.grad(out.sum(), x, create_graph=True)
    with pytest.raises(RuntimeError):
        dx.sum().backward()


# forward-mode differentiation has no rule here: a call on a dual tensor says so instead of returning a result without tangent
@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("two_step", [False, True])
def test_dual_tensors_are_refused(which, two_step):
    qkv = [torch.randn((200, 2, 64), device="cuda").to(torch.bfloat16) for _ in range(3)]
    cu = torch.tensor([0, 200], dtype=torch.int32, device="cuda")
    pattern = flash_moba.flash_topk_varlen_func(qkv[0], qkv[1], cu, cu, 200, 200, 2, 64, causal=True)
    with torch.autograd.forward_ad.dual_level():
        qkv[which] = torch.autograd.forward_ad.make_dual(qkv[which], torch.ones_like(qkv[which]))
        with pytest.raises((RuntimeError, NotImplementedError)):
            if two_step:
                flash_moba.flash_moba_attn_varlen_func(*qkv, cu, cu, 200, 200, *pattern, lg_block_m=128, lg_block_n=64, causal=True)
            else:
                flash_moba.flash_moba_varlen_func(*qkv, cu, cu, 200, 200, 64, 2)


def test_the_form_of_the_last_backward_is_reported(monkeypatch):
    def step(L, chunk, topk):
        x = [torch.randn((L, 1, 128), device="cuda").to(torch.bfloat16).requires_grad_(True) for _ in range(3)]
        cu = torch.tensor([0, L], dtype=torch.int32, device="cuda")
        seen = []
        x[0].register_hook(lambda g: seen.append(hip.last_bwd_partials()))  # (on the engine's thread, as the backward)
        flash_moba.flash_moba_varlen_func(*x, cu, cu, L, L, chunk, topk).sum().backward()
        return seen

    with monkeypatch.context() as m:
        m.setattr(hip, "host_module", lambda: _NoHost())
        assert step(8192, 128, 4) == [1] and step(512, 64, 4) == [0]
    assert step(8192, 128, 4) == [1] and step(512, 64, 4) == [0]
    with monkeypatch.context() as m:
        m.setattr(hip, "host_module", lambda: _NoHost())
        assert step(8192, 128, 4) == [1] and step(512, 64, 4) == [0]


def _csc(sel):
    """(heads, rows, chunks) bool of one sequence -> col_offsets, col_nnz, indices."""
    cn = sel.sum(1, dtype=torch.int32)
    co = cn.flatten().cumsum(0).view_as(cn).long() - cn
    return co[None].contiguous(), cn[None].contiguous(), sel.transpose(1, 2).nonzero()[:, 2].int().contiguous()


# The form, and what is allocated for it, goes by the row with the most chunks: a global token among sparse rows (the forward goes
# to row blocks, the partial rows of columns would be sized for every row by that one), rows of one density, and lists that lie in
# storage of several times their length
@pytest.mark.parametrize("D,L,chunk,others,dense,pad,rows_form", [
    (64, 4096, 64, 1, 1, 1, 1), (128, 4096, 64, 1, 1, 1, 1), (96, 4096, 128, 1, 2, 1, 1), (128, 4096, 64, 1, 0, 1, 0), (128, 2048, 64, 12, 0, 1, 1),
    (256, 2048, 64, 1, 1, 1, 0), (128, 4096, 64, 1, 0, 30, 1)])
def test_the_densest_row_decides_the_form(monkeypatch, D, L, chunk, others, dense, pad, rows_form):
    H, C = 2, L // chunk
    g = torch.Generator(device="cuda").manual_seed(D + others)
    own = (torch.arange(L, device="cuda") // chunk)[:, None]
    c = torch.arange(C, device="cuda")[None]
    sel = (c == own).repeat(H, 1, 1)
    for j in range(others):
        sel |= c == (torch.arange(L, device="cuda")[:, None] * 7 + 5 * j) % (own + 1)
    sel[:, L - 1 - torch.arange(dense, device="cuda")] = True
    sel &= c <= own
    co, cn, ind = _csc(sel)
    ind = torch.cat([ind, ind.new_zeros((pad - 1) * ind.numel())])
    cu = torch.tensor([0, L], dtype=torch.int32, device="cuda")
    q, k, v, dout = (torch.randn((L, H, D), generator=g, device="cuda").to(torch.bfloat16) for _ in range(4))

    def call():
        qg, kg, vg = (t.clone().requires_grad_(True) for t in (q, k, v))
        out = flash_moba.flash_moba_attn_varlen_func(qg, kg, vg, cu, cu, L, L, co, cn, ind, lg_block_m=128, lg_block_n=chunk, causal=True)
        res = [hip.last_fwd_row_blocks()]
        return res, (out.detach(), *torch.autograd.grad(out, (qg, kg, vg), dout))

    form, got = call()
    with monkeypatch.context() as m:
        m.setattr(hip, "host_module", lambda: _NoHost())
        _, want = call()
    assert form == [rows_form]
    for x, y in zip(got, want):
        if pad == 1:
            assert torch.equal(x, y)
        else:  # (another form of the same sums: a partial result or two of a row are rounded to bf16 in one of them)
            assert (x.float() - y.float()).norm() <= 2.0 ** -7 * y.float().norm()


def _step_with_hooks(pack, unpack, seed=5, make=None):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = [torch.randn((700, 4, 64), generator=g, device="cuda").to(torch.bfloat16) for _ in range(4)]
    q, k, v = (t.clone().requires_grad_(True) for t in x[:3])
    cu = torch.tensor([0, 300, 700], dtype=torch.int32, device="cuda")
    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
        out = flash_moba.flash_moba_varlen_func(q, k, v, cu, cu, 400, 400, 64, 3)
    return (out.detach(), *torch.autograd.grad(out, (q, k, v), x[3]))


def _spread(t):
    """The same values with twice the distance between rows, at an address that is no multiple of 16."""
    if t.dim() != 3 or t.dtype != torch.bfloat16:
        return t
    buf = torch.empty((t.shape[0], 2 * t.shape[1], t.shape[2] + 4), dtype=t.dtype, device=t.device)
    return buf[:, ::2, 4:].copy_(t)


# tensors that come back from saved-tensor hooks: anywhere in memory and with any strides they give the same gradients,
# on the CPU, in another type or in another shape they are refused (their addresses would go to kernels)
def test_saved_tensor_hooks():
    want = _step_with_hooks(lambda t: t, lambda t: t)
    for pack, unpack in ((lambda t: t.cpu(), lambda t: t.cuda()), (lambda t: t, _spread), (lambda t: t.clone(), lambda t: t)):
        assert all(torch.equal(x, y) for x, y in zip(_step_with_hooks(pack, unpack), want))
    with torch.autograd.graph.save_on_cpu():
        assert all(torch.equal(x, y) for x, y in zip(_step_with_hooks(lambda t: t, lambda t: t), want))


@pytest.mark.parametrize("unpack", [lambda t: t.cpu(), lambda t: t.float() if t.is_floating_point() else t, lambda t: t.long(), lambda t: t[:-1],
                                    lambda t: t.cpu() if t.dim() == 2 else t, lambda t: t[:, :1] if t.dtype == torch.int64 else t])
def test_saved_tensors_that_come_back_as_others_are_refused(unpack):
    with pytest.raises(RuntimeError):
        _step_with_hooks(lambda t: t, unpack)


def _layouts(name, q, k, v, dout):
    """The same values as views: slices of one projection, head-major storage, rows at twice their distance, one row for all."""
    T, H, D = q.shape
    if name == "packed":
        q, k, v = torch.stack((q, k, v), 1).unbind(1)
        dout = torch.stack((dout, dout), 1)[:, 1]
    elif name == "head_major":
        q, k, v, dout = (t.transpose(0, 1).contiguous().transpose(0, 1) for t in (q, k, v, dout))
    elif name == "spread":
        q, k, v, dout = (torch.cat((t, t), 2)[:, :, D:] for t in (q, k, v, dout))
    elif name == "expanded":  # (a gradient of stride 0, as a sum leaves it)
        dout = dout[:1, :, :1].expand(T, H, D)
    return q, k, v, dout


# strides of every kind give the bits of the packed call, natively and through the ops, forward and backward; and so does a call on
# another stream than the inputs were made on
@pytest.mark.parametrize("layout", ["packed", "head_major", "spread", "expanded"])
@pytest.mark.parametrize("L,H,D,chunk,topk", [(900, 4, 64, 64, 3), (8192, 2, 128, 128, 4), (700, 2, 256, 64, 3)])
@pytest.mark.parametrize("stream", [False, True])
def test_strided_inputs(monkeypatch, layout, L, H, D, chunk, topk, stream):
    g = torch.Generator(device="cuda").manual_seed(L + D)
    x = [torch.randn((L, H, D), generator=g, device="cuda").to(torch.bfloat16) for _ in range(4)]
    if layout == "expanded":
        x[3] = x[3][:1, :, :1].expand(L, H, D).contiguous()
    cu = torch.tensor([0, L // 3, L], dtype=torch.int32, device="cuda")
    where = (cu, cu, L - L // 3, L - L // 3)

    def step(q, k, v, dout):
        q, k, v = (t.detach().requires_grad_(True) for t in (q, k, v))
        out = flash_moba.flash_moba_varlen_func(q, k, v, *where, chunk, topk, causal=True)
        pattern = flash_moba.flash_topk_varlen_func(q, k, *where, topk, chunk, causal=True)
        out2 = flash_moba.flash_moba_attn_varlen_func(q, k, v, *where, *pattern, lg_block_m=128, lg_block_n=chunk, causal=True)
        return (out.detach(), *torch.autograd.grad(out, (q, k, v), dout), out2.detach(), *torch.autograd.grad(out2, (q, k, v), dout))

    want = step(*x)
    views = _layouts(layout, *x)
    s = torch.cuda.Stream() if stream else torch.cuda.current_stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = _both(monkeypatch, lambda: step(*views))
    torch.cuda.current_stream().wait_stream(s)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_inputs_off_16_bytes_stay_refused(monkeypatch):
    x = [torch.randn((300, 2, 64), device="cuda").to(torch.bfloat16) for _ in range(3)]
    cu = torch.tensor([0, 300], dtype=torch.int32, device="cuda")
    for host in (hip.host_module(), _NoHost()):
        monkeypatch.setattr(hip, "host_module", lambda: host)
        for i in range(3):
            y = [_spread(t) if i == j else t for j, t in enumerate(x)]
            with pytest.raises(RuntimeError, match="aligned"):
                flash_moba.flash_moba_varlen_func(*y, cu, cu, 300, 300, 64, 2)
