"""Passes that read large tensors past the caches: the lines of their rules, and every instance of the scoring one."""
import pytest
import torch

import test_gpu_delta_rows as delta
from flash_moba import flash_moba_hip as hip
from flash_moba.mean_pool import flash_topk_mean_pool
from test_gpu_few_rows import _fwd_args
from test_gpu_host_path import _both
import flash_moba

pytestmark = pytest.mark.gpu


# output rows of 128 MB and a little less; heads that share cache lines
@pytest.mark.parametrize("lens,D", [([5, 131067], 128), ([5, 131066], 128), ([70000, 262144 - 70000], 64), ([209716, 5], 80)])
def test_delta_of_every_row_at_the_line(lens, D):
    delta.test_delta_of_every_row(lens, 4, D, torch.bfloat16)


# keys below 256 MB in all, which as many sequences as long as the longest would not be; and no call could be
@pytest.mark.parametrize("lens,heads,dim,chunk", [([20000] + [100, 1, 0, 129] * 5, 16, 128, 128), ([9000, 77, 300], 32, 64, 64), ([30000, 50, 20000], 4, 96, 256), ([3000, 0, 200], 4, 40, 128)])
def test_plain_pooling_below_the_line(lens, heads, dim, chunk):
    T = sum(lens)
    assert T * heads * dim * 2 < 256 << 20
    g = torch.Generator(device="cuda").manual_seed(dim)
    k = torch.randn((T, heads, dim), generator=g, device="cuda").to(torch.bfloat16)
    cu = lambda n: torch.tensor([0] + torch.tensor(n).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
    got = flash_topk_mean_pool(k, cu(lens), max(lens), chunk)[0]
    alone, at = [], 0
    for n in lens:
        if n:
            alone.append(flash_topk_mean_pool(k[at:at + n], cu([n]), n, chunk)[0])
        at += n
    assert torch.equal(got, torch.cat(alone))
    for c in (0, got.shape[0] - 1):
        rows = k[:min(chunk, lens[0])] if c == 0 else k[T - ((lens[-1] - 1) % chunk + 1):]
        assert lens[-1] == 0 or (got[c].float() - rows.float().mean(0)).abs().max() <= 2.0 ** -8 * rows.float().mean(0).abs().max() + 1e-6


# decode steps over 256 MB of keys and a little more: heads of up to 64, 128 and 256, many rows in flight and few
@pytest.mark.parametrize("Hk,D,chunk", [(8, 64, 128), (8, 64, 64), (8, 128, 128), (16, 96, 128), (4, 256, 256), (4, 200, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_scores_from_large_pooling(monkeypatch, Hk, D, chunk, dtype):
    most = (256 << 20) // (Hk * D * 2)
    lens_k = [most // 2 + 3, 1, most // 4, most - most // 2 - most // 4 + 500]
    lens_q, H, topk = [1, 1, 2, 1], 2 * Hk, 6
    assert sum(lens_k) * Hk * D * 2 >= 256 << 20
    assert hip.load_library().fmoba_attn_fwd_gated_few_bytes(_fwd_args(lens_q, lens_k, H, Hk, D, chunk, topk)) > 0
    g = torch.Generator(device="cuda").manual_seed(D)
    mk = lambda n, h: torch.randn((n, h, D), generator=g, device="cuda").to(dtype)
    q, k, v = mk(sum(lens_q), H), mk(sum(lens_k), Hk), mk(sum(lens_k), Hk)
    cu = lambda n: torch.tensor([0] + torch.tensor(n).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
    _both(monkeypatch, lambda: (flash_moba.flash_moba_varlen_func(q, k, v, cu(lens_q), cu(lens_k), max(lens_q), max(lens_k), chunk, topk, causal=True).view(torch.int16),))
