"""Chunk means of keys that are too many for the caches: the bits of the same sequences pooled a few at a time."""
import pytest
import torch

from flash_moba.mean_pool import flash_topk_mean_pool

pytestmark = pytest.mark.gpu


# a little more than 256 MB of keys; chunks cut short, several rows in flight and few, wide rows and slices of a fused projection
@pytest.mark.parametrize("lens,heads,dim,chunk", [([100000, 1, 31200, 131], 8, 128, 128), ([131072 - 64, 77], 16, 64, 64), ([44000, 700], 32, 96, 256)])
@pytest.mark.parametrize("sliced", [False, True])
def test_large_batches_pool_as_small_ones(lens, heads, dim, chunk, sliced):
    T = sum(lens)
    assert T * heads * dim * 2 >= 256 << 20
    g = torch.Generator(device="cuda").manual_seed(dim)
    k = torch.randn((T, 2 if sliced else 1, heads, dim), generator=g, device="cuda", dtype=torch.float32).to(torch.bfloat16)[:, -1]
    cu = lambda n: torch.tensor([0] + torch.tensor(n).cumsum(0).tolist(), dtype=torch.int32, device="cuda")
    got = flash_topk_mean_pool(k, cu(lens), max(lens), chunk)[0]
    parts, at = [], 0
    for n in lens:  # in pieces of whole chunks
        for first in range(0, n, 64 * 256):
            m = min(64 * 256, n - first)
            parts.append(flash_topk_mean_pool(k[at + first:at + first + m], cu([m]), m, chunk)[0])
        at += n
    assert torch.equal(got, torch.cat(parts))
    rows = k[:chunk].float().mean(0)
    assert (got[0].float() - rows).abs().max() <= 2.0 ** -8 * rows.abs().max() + 1e-6
