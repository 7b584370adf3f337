"""Performance cases of the GQA flash-attention package: what its users call.

Three public entry points, over the sizes the repository's benchmark,
configurations and tests name:

* ``gqa_flash_attn`` — prompts (prefill), new tokens against a contiguous
  cache (decode, verification of a few draft tokens, chunked prefill) and
  bidirectional attention;
* ``GQAPagedAttention.forward`` — the serving layer over a paged cache: the
  new tokens' K/V are written at their slots, then every sequence attends its
  own blocks, in decode steps and in batches that mix prompt chunks with
  decode steps.

``listed()`` holds fixed cases, ``draw(rng)`` further ones of the same ranges.
Every case is a dict of plain values; ``kind`` is "attn" or "layer".
"""
from __future__ import annotations

import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.getcwd(), "gqa-flash-attn-rtx3060_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from gqa_kernels import gqa_flash_attn  # noqa: E402
from gqa_kernels.paged import GQAPagedAttention, PagedAttentionMetadata  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def _attn(name, batch, heads, kv_heads, seq_q, seq_kv, head_dim=128, dtype="bf16", causal=True, lse=False,
          layout="bhsd", room=0):
    """layout: "bhsd" contiguous tensors, "bshd" transposed views of a
    projection's (batch, seq, heads, head_dim) output.  room: K and V are
    views of a cache allocated for that many more keys."""
    return {"name": name, "kind": "attn", "batch": batch, "heads": heads, "kv_heads": kv_heads, "seq_q": seq_q,
            "seq_kv": seq_kv, "head_dim": head_dim, "dtype": dtype, "causal": causal, "lse": lse,
            "layout": layout, "room": room}


def _layer(name, heads, kv_heads, decodes, lo, hi, chunks=0, chunk=0, head_dim=128, dtype="bf16", block=16,
           pages="nhd", lens_seed=1):
    """`chunks` sequences with `chunk` new tokens each, then `decodes`
    sequences with one; the sequences' key counts (new tokens included) are
    uniform in [lo, hi], drawn from lens_seed.  pages: the storage order of a
    block, "nhd" (slots outer) or "hnd" (heads outer)."""
    return {"name": name, "kind": "layer", "heads": heads, "kv_heads": kv_heads, "decodes": decodes, "lo": lo,
            "hi": hi, "chunks": chunks, "chunk": chunk, "head_dim": head_dim, "dtype": dtype, "block": block,
            "pages": pages, "lens_seed": lens_seed}


def listed():
    return [
        # One token of one user early in a conversation: the smallest call,
        # all latency and launches.
        _attn("decode 1x2048", 1, 32, 8, 1, 2048, room=2048),
        # A batch of users who have just begun: short caches in a
        # preallocated buffer.
        _attn("decode 16x700", 16, 32, 8, 1, 700, room=324),
        # One token against a long document: the whole cache is streamed.
        _attn("decode 1x131072", 1, 32, 8, 1, 131072),
        # Verification of four draft tokens by a model with 64 query heads,
        # several users at mid-length contexts.
        _attn("verify 8x4x16384 64 heads", 8, 64, 8, 4, 16384),
        # A short prompt of no round length.
        _attn("prefill 1x333", 1, 32, 8, 333, 333, layout="bshd"),
        # An ordinary prompt, straight from the projections.
        _attn("prefill 1x2048", 1, 32, 8, 2048, 2048, layout="bshd"),
        # The longest prompt of the benchmark.
        _attn("prefill 1x16384", 1, 32, 8, 16384, 16384),
        # Several prompts on a model with 64-wide heads, in fp16, with the
        # log-sum-exp that a merge of partial attentions needs.
        _attn("prefill 3x2999 d64 fp16 lse", 3, 32, 8, 2999, 2999, head_dim=64, dtype="fp16", lse=True),
        # Bidirectional attention (an encoder or a scoring model) over a
        # batch of mid-length inputs.
        _attn("bidirectional 4x1025 fp16", 4, 32, 8, 1025, 1025, dtype="fp16", causal=False, layout="bshd"),
        # Chunked prefill: 512 new tokens of each of four users against
        # their caches.
        _attn("chunk 4x512x8192", 4, 32, 8, 512, 8192),
        # The serving layer's decode step: 32 sequences of every length, one
        # new token each, written and attended.
        _layer("layer decode 32x100-8000", 32, 8, 32, 100, 8000),
        # The serving layer's mixed step: two prompt chunks beside decode
        # steps.
        _layer("layer 2 chunks + 14 decodes", 32, 8, 14, 600, 6000, chunks=2, chunk=512),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _seconds(case):
    """A rough cost, to keep drawn cases within the largest listed one's."""
    w = work(case)
    return w["flops"] / (0.55e15 if case["head_dim"] == 64 else 0.9e15) + w["bytes"] / 4e12


def draw(rng):
    limit = _seconds(_attn("", 1, 32, 8, 16384, 16384))
    while True:
        heads, kv_heads = rng.choice([(32, 8), (32, 8), (64, 8), (16, 4), (24, 8)])
        head_dim = rng.choice([128, 128, 128, 64])
        dtype = rng.choice(["bf16", "bf16", "fp16"])
        common = {"head_dim": head_dim, "dtype": dtype}
        family = rng.choice(["decode", "prefill", "chunk", "bidirectional", "layer", "mixed"])
        layout = rng.choice(["bhsd", "bshd"])
        lse = rng.random() < 0.25
        if family == "decode":
            skv = _log_int(rng, 300, 131072)
            case = _attn("", _log_int(rng, 1, 32), heads, kv_heads, rng.choice([1, 1, 1, 2, 4, 7]), skv,
                         lse=lse, room=rng.choice([0, 8, 512]), **common)
        elif family == "prefill":
            s = _log_int(rng, 100, 16384)
            case = _attn("", rng.choice([1, 1, 2, 4]), heads, kv_heads, s, s, lse=lse, layout=layout, **common)
        elif family == "chunk":
            sq = _log_int(rng, 33, 1024)
            case = _attn("", rng.choice([1, 2, 4]), heads, kv_heads, sq, sq + _log_int(rng, 500, 32768),
                         lse=lse, room=rng.choice([0, 512]), **common)
        elif family == "bidirectional":
            s = _log_int(rng, 128, 4096)
            case = _attn("", _log_int(rng, 1, 16), heads, kv_heads, s, s, causal=False, lse=lse, layout=layout,
                         **common)
        else:
            hi = _log_int(rng, 1000, 32768)
            lo = max(64, int(hi * rng.uniform(0.02, 0.5)))
            pages = {"block": rng.choice([16, 16, 32, 64]), "pages": rng.choice(["nhd", "nhd", "hnd"]),
                     "lens_seed": rng.randrange(1 << 20)}
            if family == "layer":
                case = _layer("", heads, kv_heads, _log_int(rng, 1, 64), lo, hi, **pages, **common)
            else:
                chunk = min(lo, _log_int(rng, 64, 1024))
                case = _layer("", heads, kv_heads, rng.randrange(1, 31), lo, hi, chunks=rng.randrange(1, 5),
                              chunk=chunk, **pages, **common)
        if _seconds(case) <= limit:
            del case["name"]
            return case


def _lengths(case):
    """(query lengths, key counts) of a layer case's sequences."""
    rng = random.Random(case["lens_seed"])
    n = case["chunks"] + case["decodes"]
    return ([case["chunk"]] * case["chunks"] + [1] * case["decodes"],
            [rng.randint(case["lo"], case["hi"]) for _ in range(n)])


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _randn(gen, dtype, *shape):
    # N(0,1), as the repository's benchmark times every configuration on.
    out = torch.empty(shape, dtype=dtype, device="cuda")
    return out.normal_(generator=gen)


def _prepare_attn(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = _DTYPES[case["dtype"]]
    B, D = case["batch"], case["head_dim"]

    def tensor(heads, seq, room=0):
        if case["layout"] == "bshd":
            return _randn(gen, dt, B, seq + room, heads, D)[:, :seq].transpose(1, 2)
        return _randn(gen, dt, B, heads, seq + room, D)[:, :, :seq]

    return {"kind": "attn", "q": tensor(case["heads"], case["seq_q"]),
            "k": tensor(case["kv_heads"], case["seq_kv"], case["room"]),
            "v": tensor(case["kv_heads"], case["seq_kv"], case["room"]),
            "causal": case["causal"], "lse": case["lse"]}


def _prepare_layer(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = _DTYPES[case["dtype"]]
    H, Hkv, D, bs = case["heads"], case["kv_heads"], case["head_dim"], case["block"]
    qlens, klens = _lengths(case)
    n_blocks = [-(-n // bs) for n in klens]
    total = sum(n_blocks)
    perm = torch.randperm(total, generator=torch.Generator().manual_seed(seed)).tolist()
    table = torch.zeros(len(klens), max(n_blocks), dtype=torch.int32)
    slots, at = [], 0
    for b, (n, ql, kl) in enumerate(zip(n_blocks, qlens, klens)):
        row = perm[at:at + n]
        at += n
        table[b, :n] = torch.tensor(row, dtype=torch.int32)
        slots += [row[j // bs] * bs + j % bs for j in range(kl - ql, kl)]
    if case["pages"] == "hnd":
        cache = _randn(gen, dt, 2, total, Hkv, bs, D).transpose(2, 3)
    else:
        cache = _randn(gen, dt, 2, total, bs, Hkv, D)
    tokens = len(slots)
    md = PagedAttentionMetadata(slot_mapping=torch.tensor(slots, dtype=torch.int64).cuda(), block_tables=table.cuda(),
                                seq_lens=torch.tensor(klens, dtype=torch.int32).cuda(), max_seq_len=max(klens))
    if case["chunks"]:
        md.query_lens = qlens
    return {"kind": "layer", "layer": GQAPagedAttention(H, D, num_kv_heads=Hkv),
            "query": _randn(gen, dt, tokens, H * D), "key": _randn(gen, dt, tokens, Hkv * D),
            "value": _randn(gen, dt, tokens, Hkv * D), "cache": cache, "md": md}


def prepare(case, seed):
    return _prepare_attn(case, seed) if case["kind"] == "attn" else _prepare_layer(case, seed)


def run(state):
    if state["kind"] == "attn":
        return gqa_flash_attn(state["q"], state["k"], state["v"], causal=state["causal"], return_lse=state["lse"])
    out = state["layer"].forward(state["query"], state["key"], state["value"], state["cache"], state["md"])
    return out, state["cache"]


# ---------------------------------------------------------------------------
# Work
# ---------------------------------------------------------------------------
def _pairs(sq, skv, causal):
    """Visible (query, key) pairs: row i of sq sees keys [0, i + skv - sq]."""
    return sq * (skv - sq) + sq * (sq + 1) // 2 if causal else sq * skv


def work(case):
    H, Hkv, D = case["heads"], case["kv_heads"], case["head_dim"]
    if case["kind"] == "attn":
        B, sq, skv = case["batch"], case["seq_q"], case["seq_kv"]
        return {"bytes": 4 * D * B * (Hkv * skv + H * sq) + (4 * B * H * sq if case["lse"] else 0),
                "flops": 4 * D * B * H * _pairs(sq, skv, case["causal"])}
    qlens, klens = _lengths(case)
    tokens = sum(qlens)
    # The cached keys are read; the new ones come in as key / value, are
    # written to the cache and attended.
    return {"bytes": 4 * D * (Hkv * (sum(klens) + tokens) + H * tokens),
            "flops": 4 * D * H * sum(_pairs(a, b, True) for a, b in zip(qlens, klens))}


# ---------------------------------------------------------------------------
# Exact results and tolerances
# ---------------------------------------------------------------------------
def _exact_attention(q, k, v, causal, rows=2048):
    """q (H, Sq, D), k and v (Hkv, Skv, D) -> o (H, Sq, D), lse (H, Sq), in float64."""
    H, Sq, D = q.shape
    Hkv, Skv, _ = k.shape
    G = H // Hkv
    o = torch.empty(H, Sq, D, dtype=torch.float64, device=q.device)
    lse = torch.empty(H, Sq, dtype=torch.float64, device=q.device)
    kpos = torch.arange(Skv, device=q.device)
    for kvh in range(Hkv):
        kt, vv = k[kvh].double().t().contiguous(), v[kvh].double().contiguous()
        for g in range(G):
            h = kvh * G + g
            for r0 in range(0, Sq, rows):
                r1 = min(Sq, r0 + rows)
                s = torch.mm(q[h, r0:r1].double().contiguous(), kt) * D ** -0.5
                if causal:
                    qpos = torch.arange(r0, r1, device=q.device) + (Skv - Sq)
                    s.masked_fill_(kpos[None, :] > qpos[:, None], float("-inf"))
                lse[h, r0:r1] = torch.logsumexp(s, -1)
                o[h, r0:r1] = torch.mm(torch.softmax(s, -1), vv)
    return o, lse


def exact(case, seed):
    st = prepare(case, seed)
    if case["kind"] == "attn":
        parts = [_exact_attention(st["q"][b], st["k"][b], st["v"][b], case["causal"]) for b in range(case["batch"])]
        o = torch.stack([p[0] for p in parts])
        return (o, torch.stack([p[1] for p in parts])) if case["lse"] else o
    H, Hkv, D = case["heads"], case["kv_heads"], case["head_dim"]
    qlens, klens = _lengths(case)
    md, cache = st["md"], st["cache"]
    bs = case["block"]
    tokens = sum(qlens)
    blk, off = md.slot_mapping // bs, md.slot_mapping % bs
    cache[0][blk, off] = st["key"].view(tokens, Hkv, D)
    cache[1][blk, off] = st["value"].view(tokens, Hkv, D)
    out = torch.empty(tokens, H * D, dtype=torch.float64, device="cuda")
    t = 0
    for b, (ql, kl) in enumerate(zip(qlens, klens)):
        rows = md.block_tables[b, :-(-kl // bs)].long()
        k, v = (cache[i][rows].reshape(-1, Hkv, D)[:kl].transpose(0, 1) for i in (0, 1))
        q = st["query"][t:t + ql].view(ql, H, D).transpose(0, 1)
        out[t:t + ql] = _exact_attention(q, k, v, True)[0].transpose(0, 1).reshape(ql, H * D)
        t += ql
    return out, cache


def tolerance(case):
    # Outputs in the input type, probabilities rounded to it once: the
    # largest relative errors measured against float64, over the listed and
    # thirty drawn cases, are 2.35e-3 (one value: 6.0e-2 of the rms, in the
    # 16384-token prompt) in bf16 and 2.9e-4 (5.5e-3) in fp16; about four
    # times those.
    return {"rel": 1e-2, "max": 0.2} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 0.02}
