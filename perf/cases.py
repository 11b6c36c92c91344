"""What is timed of this library: its public functions on packed batches, as a program that uses them calls them.

A case is a dict of plain values:

    kind     "train": flash_moba_varlen_func and its backward; "infer": the same function without gradients (prefill,
             prefill of a later part of a sequence against the keys so far, decode steps); "two_step": the pattern from
             flash_topk_varlen_func, then flash_moba_attn_varlen_func over it; "two_step_train": with its backward
    lens_q   query rows of every sequence of the batch, lens_k its keys; where they differ the queries are the
             sequence's last rows
    heads    query heads, heads_k key / value heads, dim the head dimension
    chunk    keys per chunk, topk chunks a row keeps (its own among them when causal)
    packed   q, k and v are slices of one (tokens, 3, heads, dim) tensor, as a fused projection leaves them

Inputs are those of the library's benchmark: q, v and dout ~ N(0, 1), keys N(0, 1) plus a part shared by a chunk's keys.
"""
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "flash-moba_amd"))
from flash_moba import flash_moba_attn_varlen_func, flash_moba_varlen_func, flash_topk_varlen_func  # noqa: E402

_DTYPE = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _case(name, kind, lens_q, lens_k, heads, heads_k, dim, chunk, topk, dtype="bf16", causal=True, packed=False):
    c = {"name": name, "kind": kind, "lens_q": ",".join(map(str, lens_q)), "lens_k": ",".join(map(str, lens_k)), "heads": heads,
         "heads_k": heads_k, "dim": dim, "chunk": chunk, "topk": topk, "dtype": dtype, "causal": causal, "packed": packed}
    if name is None:
        del c["name"]
    return c


def _lens(text):
    return [int(x) for x in text.split(",")]


def _split(rng, tokens, batch, spread=0.7):
    """`tokens` cut into `batch` uneven lengths."""
    w = [np.exp(rng.gauss(0.0, spread)) for _ in range(batch)]
    lens = [max(1, int(tokens * x / sum(w))) for x in w]
    lens[0] += max(0, tokens - sum(lens))
    return lens


def listed():
    r = random.Random(20)
    # a packed batch of documents
    head = [2752, 13568, 12096, 13632, 9600, 3264, 5248, 5376]
    decode_k = [int(512 * 2 ** r.uniform(0, 6)) for _ in range(16)]
    docs = _split(r, 8191, 24)
    ragged = _split(r, 24571, 7)
    two = _split(r, 12037, 5)
    return [
        # the smallest call: BASELINE configuration 1 (two short sequences, forward); latency and launches count
        _case("c1_forward", "infer", [1024, 2048], [1024, 2048], 8, 8, 64, 128, 4),
        # a serving step: one new token for each of 16 requests with 512 to 32768 keys so far, grouped heads
        _case("decode", "infer", [1] * 16, decode_k, 32, 8, 128, 128, 8),
        # serving: the next 1024 tokens of long prompts against the keys so far
        _case("chunked_prefill", "infer", [1024, 1024, 777], [9216, 33000, 20000], 32, 8, 128, 128, 8),
        # prefill of one prompt
        _case("c2_prefill", "infer", [8192], [8192], 16, 16, 128, 128, 8),
        # the shortest point of the reference's own sweep, a training step in fp16
        _case("sweep4k_train", "train", [4096, 4096], [4096, 4096], 16, 16, 128, 128, 8, dtype="fp16"),
        # training on packed short documents with small heads, q, k and v from one projection
        _case("docs_d64_train", "train", docs, docs, 16, 16, 64, 64, 4, packed=True),
        # training with grouped key heads on a ragged batch
        _case("gqa_train", "train", ragged, ragged, 32, 8, 128, 128, 8),
        # training with the widest heads
        _case("d256_train", "train", [4096, 4096], [4096, 4096], 8, 8, 256, 128, 8),
        # gating and attention called one after the other, odd lengths and a head dimension between the powers of two
        _case("two_step_d96_train", "two_step_train", two, two, 16, 16, 96, 64, 8),
        # a training step on one long sequence with 32 heads
        _case("c3_train", "train", [32768], [32768], 32, 32, 128, 128, 16),
        # the headline training step (small chunks, many of them)
        _case("headline_train", "train", head, head, 16, 16, 128, 64, 32),
        # the largest, 2048 chunks in one sequence
        _case("c5_train", "train", [262144], [262144], 16, 16, 128, 128, 16),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """Serving (decode steps, later parts of prompts, whole prompts) and training over the ranges of the listed cases."""
    most = work(listed()[-1])["flops"]
    while True:
        what = rng.choice(["decode", "chunked", "prefill", "train", "train", "train", "two_step", "two_step_train"])
        dtype = rng.choice(["bf16", "bf16", "fp16"])
        dim = rng.choice([128, 128, 128, 128, 128, 64, 64, 64, 96, 80, 256])
        chunk = rng.choice([64, 128, 128, 256])
        heads = rng.choice([8, 16, 32])
        heads_k = rng.choice([heads, heads, heads // 4, heads // 8])
        topk = _log(rng, 2, 32)
        causal = True
        packed = False
        if what == "decode":
            batch = _log(rng, 1, 64)
            lens_k = [_log(rng, 256, 65536) for _ in range(batch)]
            lens_q = [1] * batch
        elif what == "chunked":
            batch = _log(rng, 1, 8)
            lens_q = [_log(rng, 128, 2048) for _ in range(batch)]
            lens_k = [n + _log(rng, 256, 65536) for n in lens_q]
        else:
            tokens = _log(rng, 1024, 262144)
            lens_q = lens_k = _split(rng, tokens, _log(rng, 1, 16))
            packed = heads == heads_k and what != "prefill" and rng.random() < 0.25
            causal = not (what.startswith("two_step") and rng.random() < 0.25)
        kind = what if what in ("train", "two_step", "two_step_train") else "infer"
        # wide heads come with short sequences
        if dim == 256 and sum(a * b for a, b in zip(lens_q, lens_k)) * heads > 4e9:
            continue
        c = _case(None, kind, lens_q, lens_k, heads, heads_k, dim, chunk, topk, dtype, causal, packed)
        # neither more products nor more scores of the gating than the largest listed case
        scores = sum(q * ((k + chunk - 1) // chunk) for q, k in zip(lens_q, lens_k)) * heads
        if work(c)["flops"] < 0.7 * most and scores < 4e9 and sum(lens_k) * heads_k * dim < 2 ** 30:
            return c


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype, dim, chunk = _DTYPE[case["dtype"]], case["dim"], case["chunk"]
    lens_q, lens_k = _lens(case["lens_q"]), _lens(case["lens_k"])

    def normal(rows, heads):
        return torch.randn((rows, heads, dim), generator=g, device="cuda", dtype=torch.float32)

    q = normal(sum(lens_q), case["heads"]).to(dtype)
    k = normal(sum(lens_k), case["heads_k"])
    pos = 0
    for n in lens_k:
        shared = 0.5 * normal((n + chunk - 1) // chunk, case["heads_k"])
        k[pos:pos + n] += shared.repeat_interleave(chunk, 0)[:n]
        pos += n
    k = k.to(dtype)
    v = normal(sum(lens_k), case["heads_k"]).to(dtype)
    if case["packed"]:
        q, k, v = torch.stack((q, k, v), dim=1).unbind(1)
    train = case["kind"].endswith("train")
    s = {"kind": case["kind"], "q": q, "k": k, "v": v, "chunk": chunk, "topk": case["topk"], "causal": case["causal"],
         "cu_q": torch.tensor([0] + list(np.cumsum(lens_q)), dtype=torch.int32, device="cuda"),
         "cu_k": torch.tensor([0] + list(np.cumsum(lens_k)), dtype=torch.int32, device="cuda"),
         "max_q": max(lens_q), "max_k": max(lens_k)}
    if train:
        s["dout"] = normal(sum(lens_q), case["heads"]).to(dtype)
        for name in "qkv":
            s[name] = s[name].detach().requires_grad_(True)
    return s


def run(s):
    q, k, v = s["q"], s["k"], s["v"]
    where = (s["cu_q"], s["cu_k"], s["max_q"], s["max_k"])
    with torch.set_grad_enabled(s["kind"].endswith("train")):
        if s["kind"].startswith("two_step"):
            with torch.no_grad():
                pattern = flash_topk_varlen_func(q, k, *where, s["topk"], s["chunk"], causal=s["causal"])
            out = flash_moba_attn_varlen_func(q, k, v, *where, *pattern, lg_block_m=256, lg_block_n=s["chunk"], causal=s["causal"])
            res = {"out": out, "pattern": list(pattern)}
        else:
            out = flash_moba_varlen_func(q, k, v, *where, s["chunk"], s["topk"], causal=s["causal"])
            res = {"out": out}
        if s["kind"].endswith("train"):
            res["dq"], res["dk"], res["dv"] = torch.autograd.grad(out, (q, k, v), s["dout"])
            res["out"] = out.detach()
    return res


def work(case):
    """Products of the scores of the gating and of the attention over the (row, key) pairs of the pattern (forward two
    products per pair, backward five); bytes of the inputs and outputs, once each."""
    chunk, topk, dim, heads, heads_k = case["chunk"], case["topk"], case["dim"], case["heads"], case["heads_k"]
    lens_q, lens_k = _lens(case["lens_q"]), _lens(case["lens_k"])
    pairs, scores, v_rows = 0, 0, 0
    for nq, nk in zip(lens_q, lens_k):
        if case["causal"]:
            pos = np.arange(nq, dtype=np.int64) + (nk - nq)
            pos = pos[pos >= 0]
            own = pos // chunk
            p = int((np.minimum(topk - 1, own) * chunk + pos % chunk + 1).sum())
            scores += int(own.sum())
        else:
            p = nq * min(nk, topk * chunk)
            scores += nq * ((nk + chunk - 1) // chunk)
        pairs += p
        v_rows += min(nk, p * (heads // heads_k))
    train = case["kind"].endswith("train")
    q_row, k_row = heads * dim * 2, heads_k * dim * 2
    size = sum(lens_q) * (2 * q_row + 4 * heads) + sum(lens_k) * k_row + v_rows * k_row
    if train:  # dout in, dq, dk, dv out
        size += sum(lens_q) * 2 * q_row + sum(lens_k) * 2 * k_row
    if case["kind"].startswith("two_step"):
        size += sum(lens_q) * heads * topk * 4
    return {"bytes": size, "flops": heads * dim * (2 * scores + (14 if train else 4) * pairs)}


def tolerance(case):
    # outputs and gradients are rounded to 16 bits from sums whose factors are; a near-tie of two chunks' scores that
    # another order of the sums decides the other way moves entries of the row lists by one place
    t = {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-3}
    if case["kind"].startswith("two_step"):
        t["differ"] = 1e-2
    return t
