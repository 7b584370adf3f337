"""Public entrypoint: choose single-pass vs split-KV path per workload.

MI355X rewrite of reference gqa_kernels/dispatch.py:14-62.  Same signature,
same asserts and the same bottom-right causal semantics; the route is sized
for the device's compute-unit count (256 on MI355X) instead of the fixed
``SM_COUNT = 28`` of the RTX 3060 version, and both routes launch hand-written
HIP kernels through the C ABI of libgqa_hip.so.
"""
from __future__ import annotations

import bisect
import functools
import itertools
import math
from dataclasses import dataclass

import torch

from . import _lib
from .gqa_split import (_counter_buffer, _counters, _decode_host, _workspace_buffer, _workspaces, decode_forward,
                        flat_forward, stream_handle)

__all__ = ["gqa_flash_attn", "Route", "choose_plan", "choose_route"]

LOG2E = math.log2(math.e)

# Packed query rows of one single-pass workgroup, and of one split-KV row block.
FWD_ROWS = 256
SPLIT_ROWS = 32
# At head_dim 128 one split-KV workgroup takes two row blocks when a kv head
# has more than one (each K/V chunk is then streamed once per 64 rows).
SPLIT_WIDE_ROWS = 64
# ... and all of them up to four (65-128 rows).
SPLIT_WIDER_ROWS = 128
# The split-KV path is taken for at most this many packed rows per kv head
# (at head_dim 128: SPLIT_WIDER_ROWS).
SPLIT_MAX_ROWS = 64
# At head_dim 128 (the decode first pass, gqa_decode_kernel) the split
# count first fills the compute units with one workgroup each (chunks of at
# least SPLIT_TILE keys), then doubles toward SPLIT_WG_PER_CU workgroups per
# CU only while chunks keep at least this many keys: a workgroup's first
# tiles and Q take 2-3 us to land, which short chunks do not amortise.
# Measured on MI355X (bf16, rotating K/V sets), one token at G = 4 (the
# 16-row first pass): 8192 keys 32 splits 11.5 us / 64 splits 11.8, 16384
# keys 16.0 / 16.7, 32768 keys 25.6 / 27.3, 65536 keys 44.0-44.3 / 45.1-45.3,
# 131072 keys 83.5-84.8 / 82.4-82.8 (so 64 only there); 16 tokens at 32768
# keys 35.7 / 41.5; 32 tokens at 32768 keys (128-row workgroups) 256
# workgroups 41 us, 512 51 us.  64-row workgroups (33-64 packed rows) need
# chunks of twice this: 16 tokens at 131072 keys 32 splits 92.2 us / 64
# 96.2 (8 tokens, 32-row workgroups: 87.7 / 88.7; 32 tokens, 128-row
# workgroups: 112.0 / 107.2).
SPLIT_WIDER_MIN_CHUNK = 2048
# Shortest key cache worth splitting (the reference's threshold, dispatch.py:37).
SPLIT_MIN_KV = 1024
# Keys per split-KV tile; a chunk is never shorter than this many tiles
# (one: at 4K-8K keys, 128-key chunks over twice the workgroups measured
# 5-8 % faster than 256-key chunks).
SPLIT_TILE = 128
SPLIT_MIN_TILES = 1
# Target workgroups per compute unit for the split-KV first pass (the kernel
# runs two per CU at once; one round of workgroups measured fastest).
SPLIT_WG_PER_CU = 2
# Packed rows per kv head up to which head_dim 64 also runs the 16-row
# LDS-DMA first pass (in 128-key steps), and with it the head_dim-128 split
# count with the doubling threshold counted in steps (SPLIT_WIDER_MIN_CHUNK
# keys of 64-key steps = twice as many keys of 128-key steps).  Measured on
# MI355X (bf16, one token unless noted, G = 4, rotating K/V sets, us):
# 32768 keys 32 splits 16.7 / 64 18.1 (register-staged pass: 20.1 at 64),
# 131072 keys 32 45.0 / 64 46.2 (47.9 at 64), B = 4 x 32768 8 45.1 / 16
# 46.5, 4 tokens at 131072 keys 32 45.7 / 64 47.1, B = 16 x 8192 2 45.7 / 4
# 46.5, 8192 keys 16 11.2 / 32 11.6.
DEC16_ROWS = 16
# Flat splits (gqa_split_flat_launch): for batches whose workgroups, at every
# power-of-two split count that gives each compute unit up to
# SPLIT_WG_PER_CU, would keep the fullest CU busy while the others idle more
# than this share of the time.  Measured on MI355X (bf16, one token, G = 4, 8
# kv heads, us, best fixed count / flat with one slot per CU): B = 5 x 8192
# keys (0.63 used) 33.9 / 32.1, B = 20 x 3000 (0.63) 47.6 / 43.2, B = 33 x 3000
# (0.52) 79.9 / 68.4, B = 9 x 3000 at head_dim 64 (0.56) 17.0 / 17.1; B = 3 x
# 8192 (0.75) 20.9 / 22.1, B = 12 x 6000 (0.75) 51.6 / 50.7, B = 7 x 2000 (0.88)
# 14.3 / 16.5, powers of two 0.2-1.5 us the other way (a workgroup that
# crosses into the next sequence drains and refills its pipeline).
FLAT_MIN_USED = 0.7
# ... and whose pieces keep this many tile steps (flat_piece_steps) for the
# start of each: 260 such batches, steps a piece and flat / fixed in the mean
# 2-4 1.07, 4-6 1.05, 6-8 0.99, 8-10 0.94, 10-16 0.92, more 0.87 (4 tokens, 5 x
# 1527 keys at head_dim 64 12.2 / 11.1, 20 x 1910 of 4 kv heads 21.7 / 20.6).
FLAT_MIN_PIECE = 8
# The short form of the single pass (gqa_fwd_short_launch: workgroups of
# SHORT_ROWS packed rows, two key tiles a step), considered for at most
# SHORT_MAX_WG_PER_CU workgroups per CU.  Its run time in us, fitted within
# 10 % to 34 shapes at head_dim 128 and 34 at 64 (64-4096 tokens, new tokens
# over caches up to 8192 keys, B = 1-8, causal and not): SHORT_BASE_US + the
# longest CU's sum of SHORT_ITEM_US + steps x the step time (_step_us).  The
# other routes' models count 64-key tile steps; OTHER_STEP_US is what those
# come to on these shapes.  Measured, us, other route
# -> short form: 333 tokens 17.0 -> 9.8, 1024 23.4 -> 17.4, 2048 42.1 -> 40.0
# (29.9 -> 25.8 at head_dim 64), 4 x 300 18.1 -> 15.9, 512 bidirectional
# 17.7 -> 11.2, 512 over 4096 keys 49.9 -> 44.7; 3000 tokens (three
# workgroups per CU) 77.4 / 80.4, 2048 bidirectional 62.2 / 66.1, 2 x 512 over 8192 keys
# 118.9 / 118.9, over 16384 224.9 / 232.0.
SHORT_ROWS = 128
SHORT_MAX_WG_PER_CU = 2
SHORT_BASE_US = 2.5
SHORT_ITEM_US = {128: 3.5, 64: 2.6}
SHORT_STEP_US = {128: (1.2, 1.8), 64: (0.86, 1.08)}
OTHER_STEP_US = {"single": {128: (1.25, 1.65), 64: (1.0, 1.0)}, "chunks": {128: 1.3, 64: 1.1}}
# Against the split-KV pass (33-128 packed rows, 17-64 at head_dim 64): the
# longest cache, in keys, that the short form streams faster is this times
# the root of its workgroups.  Measured, us, short / best split count, G = 4,
# 8 kv heads: 16 tokens, B = 1 300 keys 9.8 / 10.4, 600 11.9 / 10.7; B = 4 600
# 12.5 / 13.1, 1000 16.5 / 13.9; B = 16 1500 23.9 / 29.6, 3000 43.0 / 45.9;
# head_dim 64, 8 tokens, B = 1 600 9.1 / 10.2, 1000 12.1 / 10.3; B = 4 1000
# 12.1 / 12.5; B = 16 3000 28.1 / 30.6.
# Paged at head_dim 64 a step waits for more table reads: 8 x 7 tokens over
# 1484 keys (50 workgroups) 19.8 / 15.9.
SHORT_SPLIT_KEYS = {(128, False): 160.0, (128, True): 160.0, (64, False): 220.0, (64, True): 187.0}
# Single pass with key-range split of the heaviest causal query blocks: only
# considered while there are fewer than this many workgroups per CU, and
# taken when the modelled run time drops by at least FWD_SPLIT_GAIN.
FWD_SPLIT_MAX_WG_PER_CU = 2
FWD_SPLIT_GAIN = 0.05
# head_dim 64 under causal, contiguous, more blocks than CUs, where the model
# splits nothing: two workgroups share a CU there, so nearly all start
# together and the heaviest block, which the model deals one to a CU, ends
# last, alone on its CU.  Prompts have the heaviest of each (b, kv head) split,
# eight an XCD in all, up to so many ((b, kv head) pairs per XCD, blocks per
# CU); the blocks of a chunk over a long cache are nearly as long as each
# other, so up to (blocks per CU, keys per query).  Measured, us, whole / split,
# pairs x blocks: 8 x 35 2200 tokens 43.0 / 36.2, over 4400 keys 91.7 / 79.7;
# 8 x 64 4096 tokens 91.0 / 82.7, over 5120 keys 124.5 / 116.1, 8192 222 / 226,
# 16384 482 / 521; 8 x 79 5000 tokens 123.5 / 114.9; 16 x 18 1100 tokens 26.3 /
# 23.5; 16 x 40 2500 tokens 67.5 / 64.5; 32 x 15 900 tokens 28.3 / 26.6, over
# 1350 keys 43.1 / 44.5; 32 x 19 1200 tokens 38.3 / 39.1; 64 x 5 300 tokens 14.3
# / 16.2; 128 x 4 256 tokens 16.8 / 21.3; 512 x 1 64 tokens 16.2 / 26.2.  Where
# the model splits, its count: 12 x 29 1800 tokens 51.4 / 37.0 (5 blocks 46.2),
# 8 x 47 3000 tokens over 12000 keys 305 / 263 (8 blocks 299).
FWD_HEAD_PAIRS = ((2, 2.5), (4, 2.0))
FWD_HEAD_KV = ((1.5, 2.0), (2.5, 1.25))
# Per-work-item overhead of the single-pass kernel (first loads in flight,
# output, and for split blocks the exchange of the fp32 partial state), in
# 64-key tile steps, for the run-time model.  Calibrated on MI355X against
# measured split counts of causal prefill at 1024 and 2048 tokens (best
# measured: 8 of 16 blocks, -18 %; 8 of 32, -10 %; none at 4096).
FWD_ITEM_OVERHEAD = 8
# Added to each half of a split block in the persistent kernel's model:
# the exchange of its fp32 partial state (fitted to measured split counts
# at 512-3072 tokens, B = 1-5; the one-workgroup-per-item form at head_dim
# 64 measured best without it).
FWD_MERGE_OVERHEAD = 1
# Without a mask every block is as long, and a last round of few blocks costs
# as much as a full one (1025 keys, B = 4: 544 blocks on 256 CUs ran three
# rounds).  With at most three eighths of it used, the blocks left over run as
# two halves, dealt to the XCDs side by side after the whole blocks; up to
# four times as many where the model sees no difference (a block's halves then
# run in different rounds and do not wait for each other's state).  Measured,
# us, whole / split blocks, head_dim 128: B = 4 x 1025 98.5 / 84.9, 2 x 1300
# 70.3 / 61.7, 1 x 2304 110.4 / 91.8, 3 x 1500 124.0 / 112.7, 2 x 2100 163.1 /
# 147.7, 2800 134.7 / 125.6, 6200 629 / 581 (3 rounds), 4 x 2049 288 / 273 (4
# rounds).  With about half of it used, 3000 145.5 / 140.2, 8 x 1100 165.6 /
# 172.3 (a part-filled chip steps faster, and halves on every CU bring many
# merges); with more, 5 x 1100 104.1 / 116.  head_dim 64, two workgroups per
# CU: 4352 196.4 / 169.9, 5000 231.7 / 211.7, 2 x 2304 108.8 / 97.9, 8 x 1025
# 93.1 / 87.9, 6 x 700 40.2 / 37.2; 9 x 513 35.6 / 37.4, hence
# FWD_FILL_MERGE_OVERHEAD (tile steps of a half's merge there).
FWD_SPLIT_MAX_ROUNDS = 5
FWD_FILL_MERGE_OVERHEAD = 4
FWD_TILE = 64
# Pairs per XCD up to which the head_dim-128 single pass deals them (kDealPairs,
# gqa_params.hpp).
FWD_DEAL_PAIRS = 24
# The persistent single pass claims work dynamically only with at least this
# many items per workgroup (kFwdDynMinItemsPerWg, gqa_params.hpp); below it
# every workgroup takes a fixed list (gqa_fwd.hip item_at: XCD x's
# contiguous item range dealt to its workgroups round by round in snake
# order), which the run-time model then follows.
FWD_DYN_MIN_ITEMS_PER_WG = 8
# Key chunks (single pass over kv_splits key ranges per query block, then
# the split-KV combine): considered when there are fewer query blocks than
# compute units.  Per-item overhead (first loads, partial store) in tile
# steps; a tile step of the single pass takes ~1.65 us on MI355X, the
# combine launch ~3 us plus its read of the fp32 partials at ~5 TB/s.
CHUNK_ITEM_OVERHEAD = 12
CHUNK_MIN_TILES = 4
TILE_STEP_US = 1.65
COMBINE_LAUNCH_US = 3.0
COMBINE_BYTES_PER_US = 5.0e6
# Passes over the fp32 partials charged to the key-chunk route: written by
# the first pass, read back by the combine (fitted: 1.5).
CHUNK_PARTIAL_PASSES = 1.5

# Route kinds as the native calls number them (gqa_host.cpp).
_KIND_IDS = {"split": 0, "single": 1, "chunks": 2, "flat": 3, "short": 4}

_DTYPES = {torch.bfloat16: _lib.DTYPE_BF16, torch.float16: _lib.DTYPE_FP16}


@dataclass(frozen=True)
class Route:
    # "single", "split", "chunks" (splits: key chunks per query block),
    # "flat" (splits: slots of the flat split) or "short"
    kind: str
    splits: int = 1
    workgroups: int = 0
    fwd_split: int = 0  # single pass: query blocks per (b, kv head) run as two key halves


def _cdiv(a: int, b: int) -> int:
    return -(-a // b)


def _fwd_block_tiles(n_mblk: int, block_m: int, seq_q: int, seq_kv: int, causal: bool):
    """Key tiles of each single-pass query block (gqa_fwd.hip's key range)."""
    if not causal:
        return [max(0, _cdiv(seq_kv, FWD_TILE))] * n_mblk
    off = seq_kv - seq_q + FWD_TILE - 1  # a block's last position + 1 sees that many keys more, rounded up to tiles
    out = [max(0, (pid * block_m + off) // FWD_TILE) for pid in range(1, n_mblk)]
    if n_mblk > 0:
        out.append(max(0, (min(n_mblk * block_m, seq_q) + off) // FWD_TILE))
    return out


def fwd_split_makespan(tiles, n_split: int, n_bh: int, cu_count: int, causal: bool = True,
                       persistent: bool = True, dealt: bool = False) -> float:
    """Modelled run time (tile steps) of the single pass with the n_split
    heaviest blocks split: work items in the kernel's order (per (b, kv
    head): upper halves of the split blocks, then every block heavy-first
    with split blocks as their lower halves; not causal: unsplit blocks,
    then both halves of the last n_split), scheduled as _list_makespan
    describes (`persistent`: the head_dim-128 kernel over contiguous K/V;
    `dealt`: its pairs are dealt to the XCDs, which take theirs side by
    side)."""
    n = len(tiles)
    mo = FWD_MERGE_OVERHEAD if persistent else 0
    if not causal and n_split > 0:
        # (Pairs dealt to the XCDs: every XCD takes its pairs' items side by side.)
        per_xcd = n_bh // 8 if n_bh % 8 == 0 else 1
        mo = (FWD_MERGE_OVERHEAD if persistent else FWD_FILL_MERGE_OVERHEAD) + FWD_ITEM_OVERHEAD
        items = [t + FWD_ITEM_OVERHEAD for t in tiles[:n - n_split]]
        for half in (1, 0):
            items += [(t + half) // 2 + mo for t in reversed(tiles[n - n_split:])]
    else:
        per_xcd = n_bh // 8 if dealt and n_bh % 8 == 0 else 1
        lo = FWD_ITEM_OVERHEAD
        whole = [t + lo for t in tiles[:n - n_split]]
        mo += lo
        halves = [t // 2 + mo for t in tiles[n - n_split:]]
        items = [t - t // 2 + mo for t in reversed(tiles[n - n_split:])] if n_split else []
        items += (whole + halves)[::-1] if causal else whole + halves
    host = _lib._host
    if host is not None:
        return host.list_makespan(items, [per_xcd] * len(items), n_bh // per_xcd, cu_count, persistent,
                                  FWD_DYN_MIN_ITEMS_PER_WG)
    runs = [[c, per_xcd * len(list(k))] for c, k in itertools.groupby(items)]
    return _list_makespan(runs, n_bh // per_xcd, cu_count, persistent)


def _dealt(n_bh: int) -> bool:
    """Whether the head_dim-128 kernel deals n_bh (b, kv head) pairs to the
    XCDs (set_item_order, kDealPairs)."""
    return n_bh % 8 == 0 and 8 < n_bh <= 8 * FWD_DEAL_PAIRS


def _push_run(runs, cost, count: int) -> None:
    if count <= 0:
        return
    if runs and runs[-1][0] == cost:
        runs[-1][1] += count
    else:
        runs.append([cost, count])


def _slice_runs(runs, period: int, lo: int, cnt: int):
    """Runs of items [lo, lo + cnt) of `runs` (one period) repeated end to end."""
    out, i, off = [], 0, lo % period
    while off >= runs[i][1]:
        off -= runs[i][1]
        i += 1
    while cnt > 0:
        take = min(runs[i][1] - off, cnt)
        _push_run(out, runs[i][0], take)
        cnt -= take
        off, i = 0, (i + 1) % len(runs)
    return out


def _greedy_runs(runs, n: int) -> float:
    """Makespan of n CUs each taking the next item when free (the least
    loaded CU takes it), items in order.  A run of items of one cost c on
    loads within c of each other is dealt round-robin in load order (each
    item lands on the least loaded CU and leaves it the most loaded), so it
    is applied as whole rounds plus the remainder on the least loaded CUs."""
    loads = [0.0] * n  # ascending
    for c, k in runs:
        while k:
            if loads[-1] - loads[0] <= c:
                full, rem = divmod(k, n)
                if full:
                    loads = [x + full * c for x in loads]
                if rem:
                    loads = loads[rem:] + [x + c for x in loads[:rem]]
                break
            bisect.insort(loads, loads.pop(0) + c)
            k -= 1
    return loads[-1]


def _list_makespan(runs, n_rep: int, cu_count: int, persistent: bool = False) -> float:
    """Run time (tile steps) of the items of one (b, kv head), given as runs
    [cost, count] in the kernel's item order, repeated for n_rep (b, kv head)
    pairs: each XCD (cu_count / 8 CUs) takes its contiguous share of the
    whole list.  The persistent kernel with fewer than
    FWD_DYN_MIN_ITEMS_PER_WG items per workgroup deals fixed lists:
    workgroup `slot` of XCD x takes items slot, 2 S - 1 - slot, 2 S + slot,
    ... of the XCD's share (S workgroups on the XCD: gqa_fwd.hip item_at).
    Otherwise (the dynamic schedule, or one workgroup per item) each CU
    takes the next item when free.  XCD shares with the same start within
    the period and the same length are scheduled once (with 8 kv heads
    every XCD's share is the same list).  Natively once the bindings are
    loaded (gqa_host.cpp, the same steps: a plan of a new shape asks for about
    twenty of these, 0.4 ms in Python)."""
    host = _lib._host
    if host is not None:
        return host.list_makespan([c for c, _ in runs], [k for _, k in runs], n_rep, cu_count, persistent,
                                  FWD_DYN_MIN_ITEMS_PER_WG)
    period = sum(k for _, k in runs)
    total = period * n_rep
    if total == 0:
        return 0.0
    n_wg = min(total, cu_count)
    q, r = divmod(total, 8)
    static = persistent and total < FWD_DYN_MIN_ITEMS_PER_WG * n_wg
    flat = [c for c, k in runs for _ in range(k)] if static else None
    per_xcd = max(1, cu_count // 8)
    seen = {}
    worst = 0.0
    for x in range(8):
        lo, cnt = x * q + min(x, r), q + (1 if x < r else 0)
        slots = (n_wg - x + 7) >> 3
        key = (lo % period, cnt, slots if static else 0)
        if key in seen or cnt == 0:
            continue
        if static:
            # Rows of `slots` items, odd rows reversed (right-aligned when
            # short): workgroup `slot` sums column `slot`.
            share = (flat * (-(-(lo % period + cnt) // period)))[lo % period:lo % period + cnt]
            rows = []
            for j, i in enumerate(range(0, cnt, slots)):
                row = share[i:i + slots]
                pad = [0] * (slots - len(row))
                rows.append(pad + row[::-1] if j & 1 else row + pad)
            t_x = float(max(map(sum, zip(*rows))))
        else:
            t_x = _greedy_runs(_slice_runs(runs, period, lo, cnt), per_xcd)
        seen[key] = t_x
        worst = max(worst, t_x)
    return worst


def chunks_makespan(tiles, kv_splits: int, n_bh: int, cu_count: int, rows: int, head_dim: int,
                    causal: bool = True, persistent: bool = None) -> float:
    """Modelled run time (tile steps) of the single pass over key chunks:
    items (b, kv head) x chunk x query block (heavy first under causal),
    chunk c covering tiles [c * ct, (c + 1) * ct) of its block's range, plus
    the combine (launch and its read of rows x kv_splits partials).
    `persistent` (default: head_dim 128): the persistent kernel over
    contiguous K/V; paged caches run one workgroup per item."""
    n = len(tiles)
    ct = max(1, -(-max(tiles) // kv_splits))
    order = list(range(n - 1, -1, -1)) if causal else list(range(n))
    # Chunks below every block's end are full (ct tiles), chunks past every
    # block's end are empty; only the ones between differ per block.
    n_full = min(kv_splits, min(tiles) // ct)
    n_busy = min(kv_splits, -(-max(tiles) // ct))
    runs = []
    _push_run(runs, ct + CHUNK_ITEM_OVERHEAD, n_full * n)
    for c in range(n_full, n_busy):
        for m in order:
            _push_run(runs, min(ct, max(tiles[m] - c * ct, 0)) + CHUNK_ITEM_OVERHEAD, 1)
    _push_run(runs, CHUNK_ITEM_OVERHEAD, (kv_splits - n_busy) * n)
    if persistent is None:
        persistent = head_dim == 128
    first = _list_makespan(runs, n_bh, cu_count, persistent)
    # The fp32 partials are written by the first pass and read back by the
    # combine launch, each at about COMBINE_BYTES_PER_US.
    combine_us = COMBINE_LAUNCH_US + CHUNK_PARTIAL_PASSES * rows * kv_splits * (head_dim + 2) * 4 / COMBINE_BYTES_PER_US
    return first + combine_us / TILE_STEP_US


def choose_kv_chunks(batch: int, num_heads: int, num_kv_heads: int, seq_q: int, seq_kv: int,
                     cu_count: int, causal: bool, head_dim: int = 128, base: float = None,
                     persistent: bool = None) -> int:
    """Key chunks per query block for the single pass (0: none).

    With fewer query blocks than compute units (chunked prefill or a long
    verify step against a long cache) most CUs would idle; splitting every
    block's key range into kv_splits chunks (a power of two, each at least
    CHUNK_MIN_TILES tiles) fills them, at the cost of the fp32 partials and
    the combine launch.  Taken when the model beats the single pass (`base`:
    its modelled time) by FWD_SPLIT_GAIN.  `persistent` as chunks_makespan
    (False for paged caches)."""
    group = num_heads // num_kv_heads
    block_m = max(1, FWD_ROWS // group)
    n_mblk = _cdiv(seq_q, block_m)
    n_bh = batch * num_kv_heads
    if n_mblk * n_bh >= cu_count or seq_q == 0:
        return 0
    tiles = _fwd_block_tiles(n_mblk, block_m, seq_q, seq_kv, causal)
    if persistent is None:
        persistent = head_dim == 128
    if base is None:
        base = fwd_split_makespan(tiles, 0, n_bh, cu_count, causal, persistent=persistent)
    rows = batch * num_heads * seq_q
    best, best_s = base, 0
    s = 2
    while s <= _lib.GQA_MAX_SPLITS and -(-max(tiles) // s) >= CHUNK_MIN_TILES:
        t = chunks_makespan(tiles, s, n_bh, cu_count, rows, head_dim, causal, persistent)
        if t < best:
            best, best_s = t, s
        s *= 2
    return best_s if best <= (1.0 - FWD_SPLIT_GAIN) * base else 0


def _fill_last_round(n_mblk: int, n_bh: int, seq_kv: int, cu_count: int, head_dim: int) -> int:
    """Blocks per (b, kv head) whose halves fill the last round of a call
    without a mask (FWD_SPLIT_MAX_ROUNDS), or 0."""
    per_xcd, wgs = n_bh // 8, cu_count * (1 if head_dim == 128 else 2)
    if n_bh % 8 or cu_count < 8 or not wgs < n_mblk * n_bh <= FWD_SPLIT_MAX_ROUNDS * wgs:
        return 0
    left = per_xcd * n_mblk % (wgs // 8)  # blocks per XCD in the last round
    if left == 0 or left > 3 * wgs // 64:
        return 0
    tiles = [_cdiv(seq_kv, FWD_TILE)] * n_mblk
    base, *times = (fwd_split_makespan(tiles, s * _cdiv(left, per_xcd), n_bh, wgs, False, persistent=head_dim == 128)
                    for s in range(5) if s * _cdiv(left, per_xcd) <= n_mblk)
    best = min(times)
    last = max(i for i, t in enumerate(times) if t == best)
    return (last + 1) * _cdiv(left, per_xcd) if best <= (1.0 - FWD_SPLIT_GAIN) * base else 0


def choose_fwd_split(batch: int, num_heads: int, num_kv_heads: int, seq_q: int, seq_kv: int,
                     cu_count: int, causal: bool, head_dim: int = 128, persistent: bool = None,
                     dealt: bool = False) -> int:
    """Query blocks per (b, kv head) to run as two key halves (0: none).

    Under causal, when there are few workgroups per CU, the longest block
    sets the run time, and splitting the heaviest ones shortens it
    (fwd_split_makespan picks the count).  Not causal: FWD_SPLIT_MAX_ROUNDS.
    `persistent` (default: head_dim 128) and `dealt` as fwd_split_makespan;
    persistent False for paged caches."""
    group = num_heads // num_kv_heads
    block_m = max(1, FWD_ROWS // group)
    n_mblk = _cdiv(seq_q, block_m)
    n_bh = batch * num_kv_heads
    if not causal:
        return _fill_last_round(n_mblk, n_bh, seq_kv, cu_count, head_dim) if persistent is None else 0
    if n_mblk < 2:
        return 0
    whole = persistent is None and head_dim == 64  # two workgroups per CU, contiguous
    if persistent is None:
        persistent = head_dim == 128
    if n_mblk * n_bh < FWD_SPLIT_MAX_WG_PER_CU * cu_count:
        tiles = _fwd_block_tiles(n_mblk, block_m, seq_q, seq_kv, causal)
        base = fwd_split_makespan(tiles, 0, n_bh, cu_count, persistent=persistent, dealt=dealt)
        best, best_ns, last = base, 0, 0
        for f in (0.1, 0.15, 0.2, 0.25, 0.375, 0.5, 0.625, 0.75, 1.0):
            ns = max(1, min(n_mblk, round(n_mblk * f)))
            # (No shorter than its longest item: the heaviest whole block.)
            if ns == last or (ns < n_mblk and tiles[n_mblk - 1 - ns] + FWD_ITEM_OVERHEAD >= best):
                continue
            last = ns
            t = fwd_split_makespan(tiles, ns, n_bh, cu_count, persistent=persistent, dealt=dealt)
            if t < best:
                best, best_ns = t, ns
        if best <= (1.0 - FWD_SPLIT_GAIN) * base:
            return best_ns
    if whole and cu_count >= 8 and _split_head(n_mblk * n_bh / cu_count, n_bh / 8, seq_kv / seq_q):
        return min(n_mblk, max(1, round(cu_count / 4 / n_bh)))
    return 0


def _split_head(per_cu: float, pairs: float, kv_ratio: float) -> bool:
    """FWD_HEAD_PAIRS, FWD_HEAD_KV: blocks per CU, (b, kv head) pairs per XCD,
    keys per query."""
    return (per_cu > 1 and any(pairs <= p and per_cu <= c for p, c in FWD_HEAD_PAIRS)
            and any(per_cu <= c and kv_ratio <= k for c, k in FWD_HEAD_KV))


def split_rows_per_workgroup(rows: int, head_dim: int = 128) -> int:
    """Packed rows one split-KV workgroup covers (the first pass's row
    blocks: 32, or at head_dim 128 two or four of them)."""
    if head_dim != 128 or rows <= SPLIT_ROWS:
        return SPLIT_ROWS
    return SPLIT_WIDE_ROWS if rows <= SPLIT_WIDE_ROWS else SPLIT_WIDER_ROWS


def split_max_rows(head_dim: int = 128) -> int:
    """Packed rows per kv head up to which the split-KV path is taken."""
    return SPLIT_WIDER_ROWS if head_dim == 128 else SPLIT_MAX_ROWS


def split_count(base: int, seq_kv: int, cu_count: int, rows_per_wg: int, head_dim: int = 128,
                rows16: bool = False) -> int:
    """Split count of the split-KV path for `base` workgroups per split
    (head_dim 128, and head_dim 64 when the 16-row first pass runs
    (`rows16`: at most DEC16_ROWS packed rows): fill the CUs, then a second
    workgroup per CU only for chunks of SPLIT_WIDER_MIN_CHUNK keys (twice
    that for 64-row workgroups); head_dim
    64 over more rows: two workgroups per CU with chunks of SPLIT_MIN_TILES
    tiles)."""
    target = SPLIT_WG_PER_CU * cu_count
    splits = 1
    if head_dim == 128 or rows_per_wg > SPLIT_WIDE_ROWS or rows16:
        wider_min = SPLIT_WIDER_MIN_CHUNK * (2 if head_dim == 64 or rows_per_wg == SPLIT_WIDE_ROWS else 1)
        while (base * splits < cu_count and splits < _lib.GQA_MAX_SPLITS
               and _cdiv(seq_kv, splits * 2) >= SPLIT_MIN_TILES * SPLIT_TILE):
            splits *= 2
        while (base * splits < target and splits < _lib.GQA_MAX_SPLITS
               and _cdiv(seq_kv, splits * 2) >= wider_min):
            splits *= 2
        return splits
    while (base * splits < target and splits < _lib.GQA_MAX_SPLITS
           and _cdiv(seq_kv, splits * 2) >= SPLIT_MIN_TILES * SPLIT_TILE):
        splits *= 2
    return splits


def choose_route(batch: int, num_heads: int, num_kv_heads: int, seq_q: int, seq_kv: int,
                 cu_count: int, causal: bool = True, head_dim: int = 128) -> Route:
    """Pick the kernel path for one call (pure function of the shapes).

    Counterpart of reference dispatch.py:35-45.  A query block of at most
    split_max_rows(head_dim) packed rows per kv head (decode: group * seq_q = 4)
    against a cache of at least SPLIT_MIN_KV keys streams K/V with the
    split-KV kernels; the split count is a power of two: at head_dim 128
    the one that fills the compute units, doubled toward SPLIT_WG_PER_CU
    workgroups per CU while chunks keep SPLIT_WIDER_MIN_CHUNK keys; at
    head_dim 64 the one that brings the first pass to SPLIT_WG_PER_CU
    workgroups per CU, every chunk keeping at least SPLIT_MIN_TILES tiles of
    SPLIT_TILE keys (split_count).  Anything
    else (prefill, chunked prefill) runs the single-pass kernel: with a key
    split of its heaviest causal blocks (choose_fwd_split), or, when there
    are fewer query blocks than compute units, as key chunks combined by the
    split-KV combine (choose_kv_chunks, route kind "chunks") when the model
    says that is faster.
    """
    return _choose_route(batch, num_heads, num_kv_heads, seq_q, seq_kv, cu_count, causal, head_dim, False)


def _choose_route(batch, num_heads, num_kv_heads, seq_q, seq_kv, cu_count, causal, head_dim, dealt) -> Route:
    """choose_route; `dealt`: a single pass's split blocks by the model of
    dealt pairs (choose_plan)."""
    group = num_heads // num_kv_heads
    rows = group * seq_q
    single_wgs = _cdiv(seq_q, max(1, FWD_ROWS // group)) * num_kv_heads * batch
    if rows <= split_max_rows(head_dim) and seq_kv >= SPLIT_MIN_KV:
        rpw = split_rows_per_workgroup(rows, head_dim)
        base = _cdiv(rows, rpw) * num_kv_heads * batch
        splits = split_count(base, seq_kv, cu_count, rpw, head_dim, rows16=rows <= DEC16_ROWS)
        return Route("split", splits, base * splits)
    # Key chunks, against the better of the plain and the block-split single pass.
    # (Only from SPLIT_MIN_KV keys on, the length from which the reference
    # splits the key axis at all.)
    n_mblk = _cdiv(seq_q, max(1, FWD_ROWS // group))
    chunked = n_mblk * num_kv_heads * batch < cu_count and seq_q > 0 and seq_kv >= SPLIT_MIN_KV
    ns = 0
    if chunked or not dealt:
        ns = choose_fwd_split(batch, num_heads, num_kv_heads, seq_q, seq_kv, cu_count, causal, head_dim)
    if chunked:
        tiles = _fwd_block_tiles(n_mblk, max(1, FWD_ROWS // group), seq_q, seq_kv, causal)
        base = fwd_split_makespan(tiles, ns, num_kv_heads * batch, cu_count, causal, persistent=head_dim == 128)
        kc = choose_kv_chunks(batch, num_heads, num_kv_heads, seq_q, seq_kv, cu_count, causal, head_dim, base)
        if kc:
            return Route("chunks", kc, single_wgs * kc)
    if dealt:
        ns = choose_fwd_split(batch, num_heads, num_kv_heads, seq_q, seq_kv, cu_count, causal, head_dim, dealt=True)
    return Route("single", 1, single_wgs + ns * num_kv_heads * batch, ns)


def flat_steps(seq_kv: int, head_dim: int = 128) -> int:
    """Tile steps of a sequence's keys under the flat split."""
    return _cdiv(seq_kv, 128 if head_dim == 64 else 64)


def flat_piece_steps(batch: int, seq_kv: int, slots: int, head_dim: int = 128) -> float:
    """Tile steps of a piece of a flat split over `slots` ranges: every range
    is one piece, and one more for each sequence that it crosses into."""
    return batch * flat_steps(seq_kv, head_dim) / (slots + batch)


def flat_max_rows(head_dim: int = 128) -> int:
    """Packed rows per kv head up to which the flat split is built."""
    return DEC16_ROWS if head_dim == 64 else SPLIT_ROWS


def _step_us(lo: float, hi: float, work: int, longest: int, cu_count: int) -> float:
    """A step's time between `lo`, while the longest item runs with less than
    half the CUs busy on average, and `hi` with all of them."""
    return lo + (hi - lo) * min(1.0, max(0.0, 2.0 * work / (max(1, longest) * cu_count) - 1.0))


def short_us(batch: int, num_heads: int, num_kv_heads: int, seq_q: int, seq_kv: int, cu_count: int,
             causal: bool, head_dim: int = 128) -> float:
    """Modelled run time (us) of the short form (constants above): blocks
    heavy-first under causal, each CU taking the next when free."""
    block_m = SHORT_ROWS // (num_heads // num_kv_heads)
    n_mblk, n_bh = _cdiv(seq_q, block_m), batch * num_kv_heads
    tiles = _fwd_block_tiles(n_mblk, block_m, seq_q, seq_kv, causal)
    step = _step_us(*SHORT_STEP_US[head_dim], sum(tiles) * n_bh, max(tiles), cu_count)
    runs = []
    for t in (reversed(tiles) if causal else tiles):
        _push_run(runs, SHORT_ITEM_US[head_dim] + step * _cdiv(t, 2), 1)
    return SHORT_BASE_US + _list_makespan(runs, n_bh, cu_count)


def use_short(batch: int, num_heads: int, num_kv_heads: int, seq_q: int, seq_kv: int, cu_count: int,
              causal: bool, head_dim: int, kv_chunks: int, fwd_split: int, paged: bool = False) -> bool:
    """Whether the short form beats the route it would replace: the split-KV
    pass for at most split_max_rows(head_dim) packed rows per kv head, else
    the single pass with `fwd_split` split blocks, or over `kv_chunks` key
    chunks."""
    group = num_heads // num_kv_heads
    if group > SHORT_ROWS or seq_q <= 0 or batch <= 0:
        return False
    wgs = _cdiv(seq_q, SHORT_ROWS // group) * num_kv_heads * batch
    if wgs > SHORT_MAX_WG_PER_CU * cu_count:
        return False
    if group * seq_q <= split_max_rows(head_dim):
        return seq_kv <= SHORT_SPLIT_KEYS[head_dim, paged] * math.sqrt(wgs)
    block_m = max(1, FWD_ROWS // group)
    n_mblk, n_bh = _cdiv(seq_q, block_m), batch * num_kv_heads
    tiles = _fwd_block_tiles(n_mblk, block_m, seq_q, seq_kv, causal)
    persistent = head_dim == 128 and not paged
    # A second round of workgroups against one round of whole blocks of few
    # tiles, us, short / single: 15 x 74 tokens 15.6 / 13.9, 11 x 78 paged 16.1 /
    # 12.4, 15 x 54 over 64/16 heads 16.8 / 14.7; longer or split blocks gain (4 x
    # 400 19.4 / 20.7).  One tile gives the second key group nothing to do: 52 x
    # 21 paged at head_dim 64 12.2 / 10.7.
    if not kv_chunks and wgs > cu_count and (
            (head_dim == 128 and not fwd_split and n_mblk * n_bh <= cu_count and max(tiles) <= 4)
            or (head_dim == 64 and paged and max(tiles) <= 1)):
        return False
    if kv_chunks:
        other = OTHER_STEP_US["chunks"][head_dim] * chunks_makespan(
            tiles, kv_chunks, n_bh, cu_count, batch * num_heads * seq_q, head_dim, causal, persistent)
    else:
        # (The split blocks, the last fwd_split, are two items of half their tiles.)
        longest = max(max(tiles[:n_mblk - fwd_split], default=0), _cdiv(max(tiles[n_mblk - fwd_split:], default=0), 2))
        lo, hi = OTHER_STEP_US["single"][head_dim]
        other = _step_us(lo, hi, sum(tiles) * n_bh, longest, cu_count) * fwd_split_makespan(
            tiles, fwd_split, n_bh, cu_count, causal, persistent, dealt=persistent and causal and _dealt(n_bh))
    share = _short_share(kv_chunks, paged, wgs / cu_count)
    return short_us(batch, num_heads, num_kv_heads, seq_q, seq_kv, cu_count, causal, head_dim) < share * other


def _short_share(kv_chunks: int, paged: bool, wgs_per_cu: float) -> float:
    """The share of the other route's modelled time below which the short form
    is taken: what the models cannot tell apart stays with the other route.

    Key chunks are faster than their model says by up to a quarter, most when
    there are many; and a step of the short form waits for table reads when
    paged, which few workgroups do not hide.  Measured, share and short /
    chunks in us: contiguous, up to 4 chunks, 128 or more workgroups 0.95 44.7 /
    49.9, 0.96 0.83 times, fewer 0.88 37.6 / 41.4, 0.96 1.08 times, 0.98 1.29
    times; 8 chunks 0.80 22.8 / 24.9, 0.90 19.1 / 16.3, 0.99 27.0 / 21.8; paged,
    4 0.84 0.86 times, 0.90 1.05 times, 8 0.78 0.87 times, 0.91 23.0 / 16.9;
    paged with 8-28 workgroups 0.65-0.70 1.0-1.22 times.  Two paged chunks, 128
    or more workgroups, equal / unequal lengths: 0.86 146.6 / 155.7 and 114.7 /
    140.1, 0.87 132.0 / 133.8 and 111.0 / 117.5, 0.94 119.7 / 119.6 and 95.2 /
    102.5, 0.98 184.9 / 179.5 and 138.6 / 149.4."""
    if not kv_chunks:
        return 1.0
    if paged and kv_chunks == 2 and wgs_per_cu >= 0.5:
        return 0.95
    if paged or kv_chunks >= 8:
        return 0.0 if wgs_per_cu < 0.125 else 0.9 - 0.05 * paged - 0.05 * (kv_chunks >= 8)
    return 1.0 if wgs_per_cu >= 0.5 else 0.9


def choose_plan(batch: int, num_heads: int, num_kv_heads: int, seq_q: int, seq_kv: int,
                cu_count: int, causal: bool = True, head_dim: int = 128) -> Route:
    """What gqa_flash_attn launches: choose_route's route, refined.

    More than flat_max_rows(head_dim) packed rows per kv head: the short form
    of the single pass where use_short says so, and the split-KV pass for the
    remaining caches below SPLIT_MIN_KV keys.  At most that many (a token or a
    few):

    * Caches below SPLIT_MIN_KV keys are split as longer ones are (the single
      pass would give each kv head one workgroup of 256 rows, of which 4 hold
      a query): 700 keys, us, single pass / split: B = 1 20.2 / 8.7, B = 16
      20.8 / 12.7, B = 64 45.6 / 30.5; 300 keys, B = 1 14.1 / 7.4.
    * With one split per sequence the first pass writes the output itself
      (the flat split with one slot per sequence): B = 32 x 700 keys 19.5 ->
      17.6, B = 64 x 700 32.6 -> 30.5.
    * The single pass at head_dim 128 deals several (b, kv head) pairs per XCD
      side by side, which leaves less to split than choose_route's model of
      pair after pair: 2 x 1536 tokens 54.3 -> 45.4 us, 4 x 768 36.3 -> 28.9.
    * Batches that no power-of-two split count spreads evenly over the
      compute units take the flat split (FLAT_MIN_USED, FLAT_MIN_PIECE)."""
    rows = num_heads // num_kv_heads * seq_q
    if not 0 < rows <= flat_max_rows(head_dim) or seq_kv <= 0 or batch <= 0:
        route = _choose_route(batch, num_heads, num_kv_heads, seq_q, seq_kv, cu_count, causal, head_dim,
                              causal and head_dim == 128 and _dealt(batch * num_kv_heads))
        if rows <= 0 or seq_kv <= 0 or batch <= 0:
            return route
        if use_short(batch, num_heads, num_kv_heads, seq_q, seq_kv, cu_count, causal, head_dim,
                     route.splits if route.kind == "chunks" else 0, route.fwd_split):
            wgs = _cdiv(seq_q, SHORT_ROWS // (num_heads // num_kv_heads)) * num_kv_heads * batch
            return Route("short", 1, wgs)
        if rows > split_max_rows(head_dim):
            return route
    rpw = split_rows_per_workgroup(rows, head_dim)
    base = _cdiv(rows, rpw) * num_kv_heads * batch
    splits = split_count(base, seq_kv, cu_count, rpw, head_dim, rows16=rows <= DEC16_ROWS)
    if rows > flat_max_rows(head_dim):
        return Route("split", splits, base * splits)

    def used(wgs: int) -> float:
        return wgs / (cu_count * _cdiv(wgs, cu_count))

    slots = max(1, cu_count // num_kv_heads)
    if (batch > 1 and slots <= _lib.GQA_MAX_SPLITS and used(base * splits) < FLAT_MIN_USED and base * splits > cu_count
            and flat_piece_steps(batch, seq_kv, slots, head_dim) >= FLAT_MIN_PIECE):
        return Route("flat", slots, slots * num_kv_heads)
    if splits == 1 and batch <= _lib.GQA_MAX_SPLITS:
        return Route("flat", batch, base)
    return Route("split", splits, base * splits)


_route_cached = functools.lru_cache(maxsize=4096)(choose_route)
_plan_cached = functools.lru_cache(maxsize=4096)(choose_plan)


@functools.lru_cache(maxsize=None)
def _cu_count(device_index: int) -> int:
    n = _lib.load().gqa_device_cu_count(device_index)
    if n <= 0:
        raise RuntimeError(f"gqa_device_cu_count({device_index}) failed: {n}")
    return n


def _is_kernel_ready(t: torch.Tensor) -> bool:
    """The kernels need a unit last-dim stride and 16-byte aligned rows."""
    st = t.stride()
    # 16-byte alignment of the pointer and of every stride in bytes, in one
    # test (a multiple of 16 has its low four bits clear).
    return st[3] == 1 and (t.data_ptr() | ((st[0] | st[1] | st[2]) * t.element_size())) % 16 == 0


def _kernel_ready(t: torch.Tensor) -> torch.Tensor:
    """t itself, or a fresh contiguous copy when the kernels cannot read it."""
    return t if _is_kernel_ready(t) else t.clone(memory_format=torch.contiguous_format)


def gqa_flash_attn(q, k, v, causal=True, *, return_lse=False):
    """GQA flash attention.

    Args:
        q: (batch, num_heads,    seq_q,  head_dim)  — fp16 or bf16
        k: (batch, num_kv_heads, seq_kv, head_dim)
        v: (batch, num_kv_heads, seq_kv, head_dim)
        causal: if True, q position i (in K coordinates: i + seq_kv - seq_q)
                attends to K positions [0, q_pos]. Works for prefill
                (seq_q == seq_kv) and decode / chunked-prefill (seq_q < seq_kv).

        return_lse: (keyword-only extension, not in the reference) also return
                the natural-log log-sum-exp of the scaled scores of every
                query row, fp32 (batch, num_heads, seq_q); -inf for a row
                with no visible key.  Two attention outputs over disjoint key
                ranges merge exactly with it (context-parallel / ring
                attention, prefix-cache composition).

    Returns:
        (batch, num_heads, seq_q, head_dim), same dtype as q; with
        return_lse=True the pair (o, lse).
    """
    host = _lib._host
    if host is not None:
        # A planned shape with every check passed, natively; else None.
        out = host.flash_attn(q, k, v, bool(causal), bool(return_lse), _workspaces, _counters)
        if out is not None:
            return out
    batch, num_heads, seq_q, head_dim = q.shape
    _, num_kv_heads, seq_kv, _ = k.shape
    assert num_heads % num_kv_heads == 0, "num_heads must be divisible by num_kv_heads"
    assert head_dim in (64, 128), f"unsupported head_dim {head_dim}"
    assert q.is_cuda and k.is_cuda and v.is_cuda
    assert q.dtype in _DTYPES, f"unsupported dtype {q.dtype}"
    assert k.dtype == q.dtype and v.dtype == q.dtype, "q, k, v must share one dtype"
    assert v.shape == k.shape, "k and v must have the same shape"
    assert k.shape[0] == batch and k.shape[3] == head_dim, "k/v batch or head_dim differ from q"
    dev = q.get_device()  # device index (an int: no torch.device objects on this path)
    assert k.get_device() == dev and v.get_device() == dev, "q, k, v must be on one device"

    host = _decode_host()
    route = _plan_cached(batch, num_heads, num_kv_heads, seq_q, seq_kv, _cu_count(dev), bool(causal), head_dim)
    if host is not None and batch > 0 and seq_q > 0:
        host.set_plan([0, batch, num_heads, num_kv_heads, seq_q, seq_kv, head_dim, int(bool(causal)), dev, 0, 0, 0],
                      _KIND_IDS[route.kind], route.fwd_split if route.kind == "single" else route.splits,
                      (head_dim ** -0.5) * LOG2E)
        out = host.flash_attn(q, k, v, bool(causal), bool(return_lse), _workspaces, _counters)
        if out is not None:
            return out
    if dev == torch.cuda.current_device():
        return _launch(route, q, k, v, causal, return_lse, dev)
    with torch.cuda.device(dev):  # launch on q's device
        return _launch(route, q, k, v, causal, return_lse, dev)


def _base_route(q, k, causal, dev):
    batch, num_heads, seq_q, head_dim = q.shape
    return _route_cached(batch, num_heads, k.shape[1], seq_q, k.shape[2], _cu_count(dev), bool(causal), head_dim)


def _launch(route, q_in, k, v, causal, return_lse, dev):
    # One test for the usual case (all three kernel-ready; 2-byte elements:
    # the dtype is asserted), the per-tensor copies otherwise.
    qs, ks, vs = q_in.stride(), k.stride(), v.stride()
    if (qs[3] == 1 and ks[3] == 1 and vs[3] == 1
            and ((q_in.data_ptr() | k.data_ptr() | v.data_ptr()
                  | 2 * (qs[0] | qs[1] | qs[2] | ks[0] | ks[1] | ks[2] | vs[0] | vs[1] | vs[2])) & 15) == 0):
        q = q_in
    else:
        q, k, v = _kernel_ready(q_in), _kernel_ready(k), _kernel_ready(v)
    if route.kind != "single" and (k.shape[2] + 192) * max(k.stride(2), v.stride(2)) >= 1 << 30:
        # Rows so far apart that 32-bit byte offsets cannot span the keys:
        # the route by shape alone, whose split-KV pass takes them.
        route = _base_route(q, k, causal, dev)
    if route.kind == "flat":
        out = flat_forward(q, k, v, causal, route.splits, return_lse, dev)
        if out is not None:
            return out
        route = _base_route(q, k, causal, dev)
    if route.kind == "split":
        return decode_forward(q, k, v, causal, route.splits, return_lse, dev)
    o = torch.empty_like(q_in)  # as dispatch.py:47; contiguous if unusable
    if not _is_kernel_ready(o):
        o = torch.empty_like(q_in, memory_format=torch.contiguous_format)
    if route.kind == "chunks":
        return chunks_forward(q, k, v, o, causal, route.splits, return_lse)
    if route.kind == "short":
        return short_forward(q, k, v, o, causal, return_lse)
    return single_pass_forward(q, k, v, o, causal, route.fwd_split, return_lse)


def single_pass_forward(q, k, v, o, causal, fwd_split=0, return_lse=False):
    """Launch the single-pass kernel on kernel-ready q, k, v and output o
    through gqa_fwd_split_launch: with fwd_split > 0 the heaviest query
    blocks run as two key halves, and the work items are scheduled across
    the XCDs dynamically (workspace and counters: _workspace_buffer,
    _counter_buffer)."""
    lib = _lib.load()
    batch, num_heads, seq_q, head_dim = q.shape
    _, num_kv_heads, seq_kv, _ = k.shape
    scale_log2 = (head_dim ** -0.5) * LOG2E
    stream = stream_handle(q.device)
    common = (batch, num_heads, num_kv_heads, seq_q, seq_kv, head_dim,
              scale_log2, int(bool(causal)), _DTYPES[q.dtype], stream)
    qkvo = (q.data_ptr(), _lib.strides(q), k.data_ptr(), _lib.strides(k),
            v.data_ptr(), _lib.strides(v), o.data_ptr(), _lib.strides(o))
    lse = torch.empty(batch, num_heads, seq_q, dtype=torch.float32, device=q.device) if return_lse else None
    # The stream's zeroed counters: split blocks' merge counters and the
    # dynamic schedule's queues (both left zero by the kernel).
    cnt = _counter_buffer(q.device, stream, lib.gqa_fwd_split_counters_count(batch, num_kv_heads, fwd_split))
    ws = None
    if fwd_split > 0:
        ws = _workspace_buffer(q.device, stream,
                               lib.gqa_fwd_split_workspace_bytes(batch, num_kv_heads, head_dim, fwd_split))
    _lib.check(lib.gqa_fwd_split_launch(*qkvo, None if lse is None else lse.data_ptr(),
                                        None if ws is None else ws.data_ptr(), cnt.data_ptr(), fwd_split, *common))
    return o if lse is None else (o, lse)


def short_forward(q, k, v, o, causal, return_lse=False):
    """Launch the short form of the single pass (gqa_fwd_short_launch) on
    kernel-ready q, k, v and output o."""
    batch, num_heads, seq_q, head_dim = q.shape
    _, num_kv_heads, seq_kv, _ = k.shape
    lse = torch.empty(batch, num_heads, seq_q, dtype=torch.float32, device=q.device) if return_lse else None
    _lib.check(_lib.load().gqa_fwd_short_launch(
        q.data_ptr(), _lib.strides(q), k.data_ptr(), _lib.strides(k), v.data_ptr(), _lib.strides(v),
        o.data_ptr(), _lib.strides(o), None if lse is None else lse.data_ptr(), batch, num_heads, num_kv_heads,
        seq_q, seq_kv, head_dim, (head_dim ** -0.5) * LOG2E, int(bool(causal)), _DTYPES[q.dtype],
        stream_handle(q.device)))
    return o if lse is None else (o, lse)


def chunks_forward(q, k, v, o, causal, kv_splits, return_lse=False):
    """Launch the single pass over key chunks on kernel-ready q, k, v and
    output o through gqa_fwd_chunks_launch: every query block runs as
    kv_splits work items over consecutive key ranges, each writing fp32
    partials into the split workspace, which the split-KV combine reduces
    into o (and lse)."""
    lib = _lib.load()
    batch, num_heads, seq_q, head_dim = q.shape
    _, num_kv_heads, seq_kv, _ = k.shape
    stream = stream_handle(q.device)
    ws = _workspace_buffer(q.device, stream,
                           lib.gqa_split_workspace_bytes(batch, num_heads, seq_q, head_dim, kv_splits))
    cnt = _counter_buffer(q.device, stream, lib.gqa_fwd_split_counters_count(batch, num_kv_heads, 0))
    lse = torch.empty(batch, num_heads, seq_q, dtype=torch.float32, device=q.device) if return_lse else None
    _lib.check(lib.gqa_fwd_chunks_launch(
        q.data_ptr(), _lib.strides(q), k.data_ptr(), _lib.strides(k), v.data_ptr(), _lib.strides(v),
        o.data_ptr(), _lib.strides(o), None if lse is None else lse.data_ptr(), ws.data_ptr(), cnt.data_ptr(),
        kv_splits, batch, num_heads, num_kv_heads, seq_q, seq_kv, head_dim, (head_dim ** -0.5) * LOG2E,
        int(bool(causal)), _DTYPES[q.dtype], stream))
    return o if lse is None else (o, lse)
