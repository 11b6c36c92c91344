"""Row-block forward of head dimensions above 128 over long walks: where a row's reference point lies, against attention in 64 bits."""
import pytest
import torch

import flash_moba
from flash_moba import flash_moba_hip as hip

pytestmark = pytest.mark.gpu

# block maxima of 64 keys each, in units of log2: falling and rising all the way, round a cycle whose steps are all 0.4 modulo 1, and
# a first block far above a climb
STEPS = {
    "fall": lambda t: -0.45 * t, "rise": lambda t: 0.45 * t, "cycle up": lambda t: (0.4 * t) % 1.0, "cycle down": lambda t: (-0.4 * t) % 1.0,
    "peak": lambda t: torch.where(t == 0, 31.0, 0.45 * (t - 1)), "valley": lambda t: torch.where(t == 0, 0.0, -200.0 - 0.3 * (t % 7)),
}


def _scored(steps, per, D, dtype):
    """Keys whose scores (of an all-ones query, times D ** -0.5, in log2 units) are steps[i] for `per` keys each: a coarse and a fine feature, so that
    16 bits hold them to 0.02."""
    raw = steps.double().repeat_interleave(per) * D ** 0.5 * 0.6931471805599453
    k = torch.zeros((raw.numel(), 1, D), dtype=torch.float64)
    k[:, 0, 0] = (raw / 64).round() * 64
    k[:, 0, 1] = raw - k[:, 0, 0]
    return k.to(dtype).cuda()


def _exact(q, k, v):
    """Attention of the last rows of a causal sequence to all of its keys, in 64 bits; out (rows, heads, dim), lse (heads, rows)."""
    n, L, scale = q.shape[0], k.shape[0], q.shape[2] ** -0.5
    out, lse = torch.empty(q.shape, dtype=torch.float64, device="cuda"), torch.empty((q.shape[1], n), dtype=torch.float64, device="cuda")
    hidden = torch.arange(L, device="cuda")[None] > torch.arange(L - n, L, device="cuda")[:, None]
    for h in range(q.shape[1]):
        s = (q[:, h].double() @ k[:, 0].double().T * scale).masked_fill(hidden, float("-inf"))
        out[:, h], lse[h] = torch.softmax(s, -1) @ v[:, 0].double(), torch.logsumexp(s, -1)
    return out, lse


def _everything(n, L, H, chunk):
    """Lists that hold every row in every chunk that it sees."""
    C = -(-L // chunk)
    first = [max(0, c * chunk - (L - n)) for c in range(C)]
    nnz = torch.tensor([n - f for f in first], dtype=torch.int32).expand(1, H, C).contiguous()
    off = (torch.cumsum(nnz.flatten().long(), 0) - nnz.flatten()).view(1, H, C)
    rows = torch.cat([torch.arange(f, n, dtype=torch.int32) for f in first]).repeat(H)
    return off.cuda(), nnz.cuda(), rows.cuda()


def _forward(q, k, v, pattern, chunk, mode):
    n, L = q.shape[0], k.shape[0]
    cu_q, cu_k = (torch.tensor([0, x], dtype=torch.int32, device="cuda") for x in (n, L))
    out, lse, _, _ = hip.moba_varlen_fwd(q, k, v, None, *pattern, cu_q, cu_k, None, None, None, n, L, 0.0, q.shape[2] ** -0.5, False, True, 0.0, False, 128,
                                         chunk, None, _fwd_mode=mode)
    assert hip.last_fwd_row_blocks() == (mode == 2)
    return out, lse


def _assert_rounded_twice(out, exact, dtype, keys):
    """Values between 1/2 and 3/2: every probability is rounded to 16 bits once and so is the result, by half a unit in the last place each (and 1/32 of that
    for the 32-bit sums); in fp16 a probability below 2^-14 by up to 2^-25, of a sum that is at least 2^-1/2."""
    half = 2.0 ** (-9 if dtype == torch.bfloat16 else -11)
    small = 0.0 if dtype == torch.bfloat16 else keys * 2.0 ** -25 * 2 ** 0.5 * 3
    worst = ((out.double() - exact).abs() / exact).max().item()
    assert worst <= 2 * half * (1 + 2 ** -5) + small, worst


@pytest.mark.parametrize("kind", sorted(STEPS))
@pytest.mark.parametrize("steps", [64, 128, 512])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_long_walks(kind, steps, dtype):
    n, D, chunk = 33, 256, 64
    g = torch.Generator(device="cuda").manual_seed(steps)
    k = _scored(STEPS[kind](torch.arange(steps, dtype=torch.float32)), 64, D, dtype)
    v = (torch.rand(k.shape, generator=g, device="cuda") + 0.5).to(dtype)
    q = torch.ones((n, 2, D), dtype=dtype, device="cuda")
    out, lse = _forward(q, k, v, _everything(n, k.shape[0], 2, chunk), chunk, 2)
    want, want_lse = _exact(q, k, v)
    _assert_rounded_twice(out, want, dtype, k.shape[0])
    assert (lse.double() - want_lse).abs().max() <= 2e-4


# the same through the public function, whose rule takes these calls to row blocks: 16 rows of 256 heads against 32768 keys in 64 chunks
@pytest.mark.parametrize("kind", sorted(STEPS))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_long_walks_of_the_fused_call(kind, dtype):
    n, H, D, chunk, C = 16, 256, 256, 512, 64
    g = torch.Generator(device="cuda").manual_seed(1)
    k = _scored(STEPS[kind](torch.arange(C * chunk // 64, dtype=torch.float32)), 64, D, dtype)
    v = (torch.rand(k.shape, generator=g, device="cuda") + 0.5).to(dtype)
    q = torch.ones((n, H, D), dtype=dtype, device="cuda")
    cu_q, cu_k = (torch.tensor([0, x], dtype=torch.int32, device="cuda") for x in (n, C * chunk))
    out = flash_moba.flash_moba_varlen_func(q, k, v, cu_q, cu_k, n, C * chunk, chunk, C, causal=True)
    assert hip.last_fwd_row_blocks()
    want, _ = _exact(q[:, :1], k, v)
    _assert_rounded_twice(out, want.expand(n, H, D), dtype, C * chunk)


# ordinary inputs: the error against 64 bits is that of the columns, whose blocks have their own maximum for reference (1 % for the sample)
@pytest.mark.parametrize("chunk", [512, 1024])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_long_walks_are_as_precise_as_columns(chunk, dtype):
    n, H, D, C = 64, 4, 256, 64
    g = torch.Generator(device="cuda").manual_seed(chunk)
    q, k, v = (torch.randn((x, h, D), generator=g, device="cuda").to(dtype) for x, h in ((n, H), (C * chunk, 1), (C * chunk, 1)))
    pattern = _everything(n, C * chunk, H, chunk)
    want, want_lse = _exact(q, k, v)
    err = []
    for mode in (2, 1):
        out, lse = _forward(q, k, v, pattern, chunk, mode)
        err.append((float((out.double() - want).norm()), float((lse.double() - want_lse).abs().max())))
    assert err[0][0] <= err[1][0] * 1.01, err
    assert err[0][1] <= 1e-4, err
