#!/usr/bin/env python3
"""Benchmark of the MI355X GQA flash-attention forward (gqa_flash_attn).

Prints ONE JSON line (rank 0).  The headline ``value`` is causal-prefill
TFLOP/s at the Llama-3.1-8B GQA shape, seq 16384 (B=1, Hq=32, Hkv=8, D=128,
bf16); the ``decode`` object carries split-KV decode at seq_kv 131072
(microseconds and HBM GB/s), ``paged_decode`` the same decode over a paged
KV cache (gqa_kernels.paged) at two block sizes / in-block layouts,
``paged_prefill`` the chunked-prefill shape over a paged cache (and
chunks over 16384-key paged prefixes), and
``configs`` every BASELINE config (prefill 2048-16384, decode 2048-131072,
chunked prefill, the 70B decode shape) with its time and the fraction of the
roofline (MFMA or HBM) that bounds it, ``extras`` the same for a 16-token
verify step and a 128-token chunk against 131072 keys; HBM-bound configs rotate K/V sets so
the Infinity Cache cannot serve a call from the previous one.  Timing
follows reference benchmark/run.py:140-154 (untimed warm-up calls, then
back-to-back calls of the full public function between two events on the
launch stream, mean per call).  Inputs: q, k, v ~ N(0,1) from a CPU
generator seeded 0 (drawn in that order in fp32, rounded to bf16); the
headline is also timed on the reference benchmark's N(0,1) x 0.1 inputs
(``reference_benchmark_inputs``), before the headline leg.

Work counts (algorithmic, implementation overhead excluded):
  FLOPs = 4 * D * B * Hq * visible (query, key) pairs
  bytes = 2 * D * (2 * B * Hkv * Skv + 2 * B * Hq * Sq)   (K, V read; Q read, O written)

``cpu_baseline`` times the repo's CPU oracle (a numpy restatement of the
reference's torch oracle, the reference's only CPU path) on a bounded sample
of the same prefill workload, on this host's cores.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--skip-cpu] [--only WORKLOAD]
                       [--config NAME]
"""
from __future__ import annotations

import argparse
import json
import math
import os
import platform
import sys
import time
from pathlib import Path

REPO = Path(__file__).resolve().parent
sys.path.insert(0, str(REPO / "gqa-flash-attn-rtx3060_amd"))
sys.path.insert(0, str(REPO))

METRIC = "prefill TFLOP/s + decode µs & HBM GB/s, Llama-3.1-8B GQA shape, 1 MI355X"
PEAK_BF16_TFLOPS = 2516.6  # dense bf16 MFMA, 256 CU x 2.4 GHz x 4096 flop/CU/clk
PEAK_HBM_GBS = 8000.0
# Published reference number for this workload (RTX 3060, README.md:20,
# benchmark/results/rtx3060_median5.json:31): prefill 16384 in 96.195 ms.
REF_PREFILL_16K_MS = 96.195

B, HQ, HKV, D = 1, 32, 8, 128
# Inputs of every timed config: q, then k, then v drawn as N(0,1) fp32 from
# torch.Generator('cpu').manual_seed(0), rounded to bf16, copied to the GPU
# (the same bits the CPU oracle sees).  The reference benchmark times N(0,1)
# x 0.1 draws (benchmark/run.py:52-54); the headline is also timed on those
# and reported beside it (``reference_benchmark_inputs``): the shader clock
# under sustained MFMA load depends on the operands (smaller values toggle
# fewer bits and draw less power), the cycle counts do not.
REF_BENCH_SCALE = 0.1
# Tensors above this many elements (the 70B decode shape's 1 GiB K and V) are
# drawn N(0,1) on the GPU instead: a CPU draw of one takes ~10 s.
CPU_DRAW_MAX_ELEMS = 1 << 28
PREFILL_S = 16384
DECODE_S = 131072


def visible_pairs(sq: int, skv: int, causal: bool = True) -> int:
    """Unmasked (query, key) pairs per (batch, head): row i sees keys
    [0, i + skv - sq], clipped to [0, skv) (bottom-right causal)."""
    import numpy as np
    if not causal:
        return sq * skv
    return int(np.clip(np.arange(sq, dtype=np.int64) + (skv - sq) + 1, 0, skv).sum())


def flops(b, hq, sq, skv, d, causal=True) -> int:
    return 4 * d * b * hq * visible_pairs(sq, skv, causal)


def hbm_bytes(b, hq, hkv, sq, skv, d, elem=2) -> int:
    return elem * d * (2 * b * hkv * skv + 2 * b * hq * sq)


def _inputs(torch, b, hq, hkv, sq, skv, d, n_kv_sets=1, scale=1.0, dtype=None):
    """q and n_kv_sets (k, v) pairs on the GPU, bf16 unless `dtype` says
    otherwise.  q and the first k, v are N(0,1) draws (times `scale`) from a
    CPU generator seeded 0, in the order q, k, v, rounded from fp32.  The
    further K/V sets, which only keep consecutive calls of an HBM-bound
    config from finding their keys in the Infinity Cache, and tensors above
    CPU_DRAW_MAX_ELEMS come from a seeded GPU generator (also N(0,1) times
    `scale`)."""
    dt = torch.bfloat16 if dtype is None else dtype
    g = torch.Generator(device="cpu").manual_seed(0)
    gg = torch.Generator(device="cuda").manual_seed(1)

    def draw(shape, cpu):
        if cpu and math.prod(shape) <= CPU_DRAW_MAX_ELEMS:
            return (torch.randn(shape, generator=g) * scale).to(dt).to("cuda")
        return (torch.randn(shape, device="cuda", generator=gg) * scale).to(dt)

    q = draw((b, hq, sq, d), True)
    kvs = [(draw((b, hkv, skv, d), i == 0), draw((b, hkv, skv, d), i == 0)) for i in range(n_kv_sets)]
    return q, kvs


INPUTS_NOTE = ("synthetic N(0,1): q, k, v drawn in that order from torch.Generator('cpu').manual_seed(0) "
               "in fp32, rounded to bf16 (extra rotating K/V sets of HBM-bound configs and the 70B "
               "shape's 1 GiB K/V: N(0,1) from a seeded GPU generator); reference_benchmark_inputs: "
               "the headline on the reference benchmark's N(0,1) x 0.1 inputs")


def _time(torch, fn, steps, warmup, warm_ms=0.0):
    """Mean ms per call of fn() over `steps` back-to-back calls, timed with
    events on torch's current stream (the stream the kernels launch on),
    after `warmup` untimed calls; with warm_ms > 0 the untimed calls go on
    until that much wall time has passed (the shader clock ramps down while
    the GPU idles, e.g. while the host draws the next inputs, and takes tens
    of milliseconds of load to come back)."""
    for _ in range(warmup):
        fn(0)
    torch.cuda.synchronize()
    if warm_ms > 0:
        # (rotating the call index as the timed calls do, so that a config
        # that rotates K/V sets meets the Infinity Cache in its steady state)
        t_end = time.perf_counter() + warm_ms * 1e-3
        j = 0
        while time.perf_counter() < t_end:
            for _ in range(8):
                fn(j)
                j += 1
            torch.cuda.synchronize()
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record()
    for i in range(steps):
        fn(i)
    end.record()
    torch.cuda.synchronize()
    return start.elapsed_time(end) / steps


def _gate(torch, gqa_flash_attn, q, k, v, rows=64, heads=(0, 1, 2, 3, 31)):
    """Correctness gate on the timed inputs: the last `rows` query rows of a
    few heads against a plain fp32 torch computation (max/mean abs error)."""
    out = gqa_flash_attn(q, k, v, causal=True)
    sq, skv, d = q.shape[2], k.shape[2], q.shape[3]
    g = q.shape[1] // k.shape[1]
    worst_max, sum_mean = 0.0, 0.0
    for h in heads:
        qq = q[0, h, sq - rows:].float().contiguous()
        kt = k[0, h // g].float().t().contiguous()
        s = torch.matmul(qq, kt) * d ** -0.5
        qpos = torch.arange(sq - rows, sq, device="cuda") + (skv - sq)
        s.masked_fill_(qpos[:, None] < torch.arange(skv, device="cuda")[None, :], float("-inf"))
        ref = torch.matmul(torch.softmax(s, -1), v[0, h // g].float().contiguous())
        diff = (out[0, h, sq - rows:].float() - ref).abs()
        worst_max = max(worst_max, diff.max().item())
        sum_mean += diff.mean().item()
    return {"max_abs": worst_max, "mean_abs": sum_mean / len(heads), "rows_checked": rows * len(heads)}


def _cpu_threads() -> int:
    try:
        from threadpoolctl import threadpool_info
        n = [i.get("num_threads", 1) for i in threadpool_info() if i.get("user_api") == "blas"]
        if n:
            return int(max(n))
    except Exception:
        pass
    return len(os.sched_getaffinity(0))


def _cpu_model() -> str:
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return platform.processor() or "unknown"


def cpu_baseline(torch, q, k, v, budget_s=12.0):
    """Time the CPU oracle on a bounded sample of the prefill workload: the
    query group of kv head 0 (4 heads) for the last `n` rows, n doubled until
    one run takes ~budget_s/4, then median of 3 runs."""
    import numpy as np
    from oracle.gqa_oracle import gqa_reference
    sq, skv, d = q.shape[2], k.shape[2], q.shape[3]
    g = q.shape[1] // k.shape[1]
    qn = q[:, :g].float().cpu().numpy()
    kn = k[:, :1].float().cpu().numpy()
    vn = v[:, :1].float().cpu().numpy()
    n = 64
    while True:
        rows = np.arange(sq - n, sq)
        t0 = time.perf_counter()
        gqa_reference(qn, kn, vn, True, rows=rows, dtype=np.float32)
        dt = time.perf_counter() - t0
        if dt > budget_s / 4 or n >= sq:
            break
        n = min(sq, n * 4 if dt < budget_s / 32 else n * 2)
    times = [dt]
    for _ in range(2):
        t0 = time.perf_counter()
        gqa_reference(qn, kn, vn, True, rows=rows, dtype=np.float32)
        times.append(time.perf_counter() - t0)
    t = sorted(times)[1]
    work = 4 * d * g * sum(min(skv, int(r) + (skv - sq) + 1) for r in rows)
    return {
        "value": work / t / 1e12,
        "unit": "TFLOP/s",
        "cores": _cpu_threads(),
        "kind": "port",
        "sample": (f"numpy fp32 oracle, causal prefill S={sq}: q heads 0-{g - 1} (kv head 0), "
                   f"last {n} query rows ({work / 1e9:.1f} GFLOP), median of 3 runs "
                   f"({t:.2f} s each) on {_cpu_model()}"),
        "seconds_per_run": t,
    }


def cpu_decode_baseline(torch, budget_runs=10):
    """The reference's CPU config: decode B=1, Hq=32,
    Hkv=8, D=128, seq_q=1, seq_kv=2048, N(0,1) from a CPU seed-0 generator."""
    import numpy as np
    from oracle.gqa_oracle import gqa_reference
    gen = torch.Generator(device="cpu").manual_seed(0)
    q = torch.randn(1, 32, 1, 128, generator=gen).to(torch.bfloat16).float().numpy()
    k = torch.randn(1, 8, 2048, 128, generator=gen).to(torch.bfloat16).float().numpy()
    v = torch.randn(1, 8, 2048, 128, generator=gen).to(torch.bfloat16).float().numpy()
    for _ in range(3):
        gqa_reference(q, k, v, True)
    ts = []
    for _ in range(budget_runs):
        t0 = time.perf_counter_ns()
        gqa_reference(q, k, v, True)
        ts.append(time.perf_counter_ns() - t0)
    us = sorted(ts)[len(ts) // 2] / 1e3
    return {"us": us, "gbs": hbm_bytes(1, 32, 8, 1, 2048, 128) / (us * 1e-6) / 1e9,
            "cores": _cpu_threads(), "config": "decode B=1 Hq=32 Hkv=8 D=128 Sq=1 Skv=2048"}


TRAFFIC_FILE = REPO / "profiles" / "hbm_traffic.json"


def _load_traffic():
    """Measured HBM traffic per launch (rocprofv3 FETCH_SIZE / WRITE_SIZE,
    scaled by what the same counters read for a plain copy of known size),
    recorded in profiles/hbm_traffic.json; None if absent."""
    try:
        return json.loads(TRAFFIC_FILE.read_text())
    except (OSError, ValueError):
        return None


def _traffic_bytes(traffic, workload):
    if not traffic or workload not in traffic.get("workloads", {}):
        return None
    return traffic["workloads"][workload]["hbm_bytes_per_call"]


def gemm_ceiling(torch, n=16384, steps=5, warmup=2):
    """bf16 GEMM n x n x n through torch.matmul (hipBLASLt): the practical
    dense-MFMA ceiling of this GPU, for comparison with the published peak."""
    g = torch.Generator(device="cuda").manual_seed(7)
    a = torch.randn(n, n, device="cuda", generator=g).to(torch.bfloat16)
    b = torch.randn(n, n, device="cuda", generator=g).to(torch.bfloat16)
    ms = _time(torch, lambda i: torch.matmul(a, b), steps, warmup)
    del a, b
    return {"kernel": f"torch.matmul bf16 {n}x{n}x{n} (hipBLASLt)", "ms": ms,
            "tflops": 2 * n ** 3 / (ms * 1e-3) / 1e12}


def copy_calibration(torch, steps, warmup):
    """A plain device copy of 1 GiB (torch's copy kernel): reads and writes
    exactly 2^30 bytes per launch, the reference point for the HBM traffic
    counters."""
    n = 1 << 28  # fp32 elements = 1 GiB
    src = torch.empty(n, dtype=torch.float32, device="cuda").uniform_()
    dst = torch.empty_like(src)
    ms = _time(torch, lambda i: dst.copy_(src), steps, warmup)
    return {"workload": "copy 1 GiB fp32 (calibration)", "bytes_read": 4 * n, "bytes_written": 4 * n,
            "ms": ms, "gbs": 8 * n / (ms * 1e-3) / 1e9}


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--skip-cpu", action="store_true", help="omit the CPU baseline legs")
    ap.add_argument("--warm-ms", type=float, default=WARM_MS,
                    help="minimum untimed time per config beyond the headline (0: the --warmup calls only; "
                         "for counter-collection runs)")
    ap.add_argument("--config", default=None,
                    help="with --only configs (or extras): time only the configs (extra shapes) whose name starts with this")
    ap.add_argument("--only", choices=["prefill", "decode", "paged", "copy", "gemm", "chunked", "70b", "configs",
                                       "extras"],
                    default=None,
                    help="time one workload only (for profiling runs); 'copy' times a plain 1 GiB "
                         "device copy, the calibration kernel of the HBM traffic counters; 'gemm' "
                         "a 16384^3 bf16 library GEMM, the practical MFMA ceiling of the box; "
                         "'chunked' and '70b' one BASELINE config each; 'configs' every BASELINE config; "
                         "'extras' the verify-step and key-chunk shapes")
    args = ap.parse_args()

    _set_warm_ms(args.warm_ms)
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print(f"bench.py: this build measures one GPU only (asked for --gpus {args.gpus}, "
              f"WORLD_SIZE={world}); the attention path has no multi-GPU component.",
              file=sys.stderr)
        return 2

    import torch
    from gqa_kernels import gqa_flash_attn

    if not torch.cuda.is_available():
        print("bench.py: no GPU visible", file=sys.stderr)
        return 2

    result = {
        "metric": METRIC, "value": None, "unit": "TFLOP/s", "n_gpus": 1,
        "steps": args.steps, "warmup": args.warmup, "ms_per_step": None,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "bf16", "data": INPUTS_NOTE,
        "config": {"workload": f"causal GQA prefill B={B} Hq={HQ} Hkv={HKV} D={D} seq={PREFILL_S}",
                   "global_batch": B, "seq_len": PREFILL_S, "parallelism": "single GPU"},
    }

    if args.only == "copy":
        print(json.dumps(copy_calibration(torch, args.steps, args.warmup)))
        return 0
    if args.only == "gemm":
        print(json.dumps(gemm_ceiling(torch)))
        return 0

    traffic = _load_traffic()

    # ---------------- prefill (headline) ----------------
    if args.only in (None, "prefill"):
        # Both input sets are drawn first (the GPU idles meanwhile), then the
        # reference-benchmark-input leg runs, then the headline: W untimed
        # and K timed calls each.  From idle, the first ~40 ms of prefill
        # calls run ~2 % slower while the shader clock ramps up; the headline
        # leg follows another leg of the same kernel, as calls do in a
        # running service.
        q, kvs = _inputs(torch, B, HQ, HKV, PREFILL_S, PREFILL_S, D)
        k, v = kvs[0]
        q1, kvs1 = _inputs(torch, B, HQ, HKV, PREFILL_S, PREFILL_S, D, scale=REF_BENCH_SCALE)
        k1, v1 = kvs1[0]
        fl = flops(B, HQ, PREFILL_S, PREFILL_S, D)
        gate1 = _gate(torch, gqa_flash_attn, q1, k1, v1)
        ms1 = _time(torch, lambda i: gqa_flash_attn(q1, k1, v1, causal=True), args.steps, args.warmup)
        tf1 = fl / (ms1 * 1e-3) / 1e12
        del q1, k1, v1, kvs1
        gate = _gate(torch, gqa_flash_attn, q, k, v)
        ms = _time(torch, lambda i: gqa_flash_attn(q, k, v, causal=True), args.steps, args.warmup)
        tflops = fl / (ms * 1e-3) / 1e12
        result.update(value=tflops, ms_per_step=ms)
        result["vs_baseline"] = REF_PREFILL_16K_MS / ms
        result["vs_baseline_basis"] = ("speed-up over the reference's published RTX 3060 time for "
                                       f"this workload ({REF_PREFILL_16K_MS} ms)")
        result["gate"] = gate
        result["reference_benchmark_inputs"] = {
            "inputs": f"N(0,1) x {REF_BENCH_SCALE} (reference benchmark/run.py:52-54), same CPU seed-0 draws",
            "ms_per_step": ms1, "value": tf1, "frac": tf1 / PEAK_BF16_TFLOPS, "gate": gate1}
        result["roofline"] = {
            "bound": "mfma", "kernel": "gqa_fwd_kernel", "achieved": tflops,
            "peak": PEAK_BF16_TFLOPS, "unit": "TFLOP/s", "frac": tflops / PEAK_BF16_TFLOPS,
            "traffic": _traffic_bytes(traffic, "prefill"), "flops_per_launch": fl,
            "note": "achieved = algorithmic FLOPs per launch / mean launch time (one launch per step); "
                    "traffic = HBM bytes per launch from rocprofv3 FETCH_SIZE + WRITE_SIZE, "
                    "calibrated on a plain copy (" + TRAFFIC_FILE.name + ")",
        }
        if not args.skip_cpu:
            result["cpu_baseline"] = cpu_baseline(torch, q, k, v)
        del q, k, v, kvs
        torch.cuda.empty_cache()
        # Context for `peak`: what the vendor GEMM reaches on this box (the
        # shader clock runs well below the 2.4 GHz the published peak assumes
        # under sustained MFMA load).
        gemm = gemm_ceiling(torch)
        result["roofline"]["gemm_ceiling"] = gemm
        result["roofline"]["frac_of_gemm_ceiling"] = tflops / gemm["tflops"]
        torch.cuda.empty_cache()

    # ---------------- decode ----------------
    if args.only in (None, "decode"):
        # Two K/V sets (1 GiB) so consecutive calls do not hit the 256 MB
        # Infinity Cache with the previous call's data.
        q, kvs = _inputs(torch, B, HQ, HKV, 1, DECODE_S, D, n_kv_sets=2)
        dsteps = max(args.steps * 5, 50)
        ms = _time(torch, lambda i: gqa_flash_attn(q, *kvs[i % 2], causal=True), dsteps, args.warmup * 2,
                   warm_ms=WARM_MS)
        by = hbm_bytes(B, HQ, HKV, 1, DECODE_S, D)
        gbs = by / (ms * 1e-3) / 1e9
        from gqa_kernels.dispatch import _cu_count, choose_plan
        route = choose_plan(B, HQ, HKV, 1, DECODE_S, _cu_count(0), causal=True, head_dim=D)
        result["decode"] = {
            "workload": f"causal GQA decode B={B} Hq={HQ} Hkv={HKV} D={D} seq_q=1 seq_kv={DECODE_S}",
            "us": ms * 1e3, "gbs": gbs, "steps": dsteps, "splits": route.splits,
            "roofline": {"bound": "hbm", "achieved": gbs, "peak": PEAK_HBM_GBS, "unit": "GB/s",
                         "frac": gbs / PEAK_HBM_GBS, "bytes_per_call": by,
                         "traffic": _traffic_bytes(traffic, "decode"),
                         "note": "whole call (split first pass + combine), 2 rotating K/V sets; "
                                 "traffic = measured HBM bytes per call (" + TRAFFIC_FILE.name + ")"},
        }
        if not args.skip_cpu:
            result["decode"]["cpu_baseline"] = cpu_decode_baseline(torch)
        del q, kvs
        torch.cuda.empty_cache()
        # Context for `peak`: what a plain device copy (torch's copy kernel,
        # reads and writes) moves per second on this box.
        copy = copy_calibration(torch, 10, 3)
        result["decode"]["roofline"]["copy_ceiling"] = {"kernel": "torch copy_ of 1 GiB fp32 (read + write)",
                                                        "us": copy["ms"] * 1e3, "gbs": copy["gbs"]}
        result["decode"]["roofline"]["frac_of_copy_ceiling"] = gbs / copy["gbs"]
        torch.cuda.empty_cache()

    # ---------------- decode and chunked prefill over a paged KV cache ----------------
    if args.only in (None, "paged"):
        result["paged_decode"] = paged_decode(torch, max(args.steps * 5, 50), args.warmup * 2, traffic)
        torch.cuda.empty_cache()
        result["paged_prefill"] = paged_prefill(torch, args.steps, args.warmup)
        torch.cuda.empty_cache()

    # ---------------- every BASELINE config ----------------
    if args.only is None:
        result["configs"] = sweep(torch, gqa_flash_attn, args.steps, args.warmup)
        result["extras"] = sweep(torch, gqa_flash_attn, args.steps, args.warmup, table=EXTRAS)
    elif args.only == "extras":
        result["extras"] = sweep(torch, gqa_flash_attn, args.steps, args.warmup, only=args.config, table=EXTRAS)
    elif args.only in ("chunked", "70b"):
        result["configs"] = sweep(torch, gqa_flash_attn, args.steps, args.warmup,
                                  only={"chunked": "chunked", "70b": "70B"}[args.only])
    elif args.only == "configs":
        result["configs"] = sweep(torch, gqa_flash_attn, args.steps, args.warmup, only=args.config)

    if result["value"] is None and "decode" in result:
        d = result["decode"]
        result.update(value=d["gbs"], unit="GB/s", ms_per_step=d["us"] / 1e3)
        result["config"]["workload"] = d["workload"]
    print(json.dumps(result))
    return 0


def paged_decode(torch, steps, warmup, traffic=None):
    """Decode at seq_kv 131072 over a paged cache (gqa_kernels.paged): one
    line per (block size, in-block layout), blocks assigned in a random
    order, two rotating caches as for the contiguous decode."""
    from gqa_kernels.paged import paged_attention
    g = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn(B, HQ, 1, D, device="cuda", generator=g).to(torch.bfloat16)
    lens = torch.full((B,), DECODE_S, dtype=torch.int32, device="cuda")
    by = hbm_bytes(B, HQ, HKV, 1, DECODE_S, D)
    out = []
    for bs, layout in ((64, "HND"), (16, "NHD")):
        nblk = B * DECODE_S // bs
        caches = []
        for _ in range(2):
            shape = (nblk, HKV, bs, D) if layout == "HND" else (nblk, bs, HKV, D)
            kc, vc = (torch.randn(*shape, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
            if layout == "HND":
                kc, vc = kc.transpose(1, 2), vc.transpose(1, 2)
            table = torch.randperm(nblk, device="cuda", generator=g).to(torch.int32).view(B, -1)
            caches.append((kc, vc, table))
        ms = _time(torch, lambda i: paged_attention(q, *caches[i % 2], lens, True, max_seq_len=DECODE_S),
                   steps, warmup, warm_ms=WARM_MS)
        out.append({"workload": f"paged causal GQA decode B={B} Hq={HQ} Hkv={HKV} D={D} seq_q=1 "
                                f"seq_kv={DECODE_S} block_size={bs} layout={layout}",
                    "us": ms * 1e3, "gbs": by / (ms * 1e-3) / 1e9,
                    "frac_of_hbm_peak": by / (ms * 1e-3) / 1e9 / PEAK_HBM_GBS,
                    "traffic": _traffic_bytes(traffic, f"paged_bs{bs}_{layout}")})
        del caches
    return out


def paged_prefill(torch, steps, warmup):
    """The chunked-prefill BASELINE shape (B=4, 512 new tokens attending 8192
    keys, causal) over a paged cache (gqa_kernels.paged, single-pass route),
    128-key HND blocks, 64-key NHD blocks and 16-key NHD blocks (vLLM's
    default block size) in random order; then two sequences' 512-token
    chunks over 16384 keys (the single pass with split query blocks) and
    one sequence's 128-token chunk over a 16384-key prefix (the key-chunk
    route), in 16-key NHD blocks."""
    from gqa_kernels.paged import paged_attention
    out = []
    for b, sq, skv, legs in ((4, 512, 8192, ((128, "HND"), (64, "NHD"), (16, "NHD"))),
                             (2, 512, 16384, ((16, "NHD"),)),
                             (1, 128, 16384, ((16, "NHD"),))):
        out += _paged_prefill_legs(torch, paged_attention, b, sq, skv, legs, steps, warmup)
    return out


def _paged_prefill_legs(torch, paged_attention, b, sq, skv, legs, steps, warmup):
    g = torch.Generator(device="cuda").manual_seed(4)
    q = torch.randn(b, HQ, sq, D, device="cuda", generator=g).to(torch.bfloat16)
    lens = torch.full((b,), skv, dtype=torch.int32, device="cuda")
    fl = flops(b, HQ, sq, skv, D)
    out = []
    for bs, layout in legs:
        nblk = b * skv // bs
        shape = (nblk, HKV, bs, D) if layout == "HND" else (nblk, bs, HKV, D)
        kc, vc = (torch.randn(*shape, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
        if layout == "HND":
            kc, vc = kc.transpose(1, 2), vc.transpose(1, 2)
        table = torch.randperm(nblk, device="cuda", generator=g).to(torch.int32).view(b, -1)
        ms = _time(torch, lambda i: paged_attention(q, kc, vc, table, lens, True, max_seq_len=skv), steps, warmup,
                   warm_ms=WARM_MS)
        out.append({"workload": f"paged causal GQA chunked prefill B={b} Hq={HQ} Hkv={HKV} D={D} seq_q={sq} "
                                f"seq_kv={skv} block_size={bs} layout={layout}",
                    "us": ms * 1e3, "tflops": fl / (ms * 1e-3) / 1e12,
                    "frac_of_mfma_peak": fl / (ms * 1e-3) / 1e12 / PEAK_BF16_TFLOPS})
        del kc, vc
    return out


# Every BASELINE config (BASELINE.json "configs"): name, B, Hq, Hkv, seq_q,
# seq_kv, the roofline that bounds it and head_dim.  configs[0] is the
# reference's CPU config (decode at 2048 keys), here timed on the GPU beside
# its CPU time.  The last row is the 16K prefill at head_dim 64, the other
# head size the reference accepts (dispatch.py:32).
CONFIGS = (
    [("cpu-config decode 2048", 1, 32, 8, 1, 2048, "hbm", 128)]
    + [(f"prefill {s}", 1, 32, 8, s, s, "mfma", 128) for s in (2048, 4096, 8192, 16384)]
    + [(f"decode {s}", 1, 32, 8, 1, s, "hbm", 128) for s in (8192, 32768, 131072)]
    + [("chunked prefill B=4 512/8192", 4, 32, 8, 512, 8192, "mfma", 128),
       ("70B decode B=16 Hq=64 Sq=4 32768", 16, 64, 8, 4, 32768, "hbm", 128),
       ("prefill 16384 head_dim 64", 1, 32, 8, 16384, 16384, "mfma", 64)]
)
# Shapes beyond the BASELINE configs that exercise the other routes (timed
# in the default run as ``extras``): a verify step of 16 tokens (64 packed
# rows per kv head: the decode first pass with 64-row workgroups) and a
# 128-token chunk (the single pass over key chunks), both against 131072 keys;
# then the headline prefill and decode in fp16 (the other input type the
# reference accepts, dispatch.py:18) and with the LSE side output
# (return_lse=True), and the decode at head_dim 64 (dispatch.py:32).  Optional trailing fields: dtype ("bf16" default,
# "fp16") and return_lse.
EXTRAS = (
    ("verify 16 x 131072", 1, 32, 8, 16, 131072, "hbm", 128),
    ("chunk 128 x 131072", 1, 32, 8, 128, 131072, "mfma", 128),
    ("prefill 16384 fp16", 1, 32, 8, 16384, 16384, "mfma", 128, "fp16"),
    ("decode 131072 fp16", 1, 32, 8, 1, 131072, "hbm", 128, "fp16"),
    ("prefill 16384 return_lse", 1, 32, 8, 16384, 16384, "mfma", 128, "bf16", True),
    ("decode 131072 return_lse", 1, 32, 8, 1, 131072, "hbm", 128, "bf16", True),
    ("decode 131072 head_dim 64", 1, 32, 8, 1, 131072, "hbm", 64),
)
# Untimed calls of every config beyond the headline run for at least this
# long before its timed calls (its inputs were just drawn on the host, the
# GPU idle meanwhile, and the clock needs tens of milliseconds of load to
# ramp back up).
WARM_MS = 150.0


def _set_warm_ms(ms: float) -> None:
    global WARM_MS
    WARM_MS = ms
# K/V sets rotated per HBM-bound config: enough that consecutive calls cannot
# find the previous calls' keys in the 256 MB Infinity Cache.
ROTATE_BYTES = 600e6


def sweep(torch, gqa_flash_attn, steps=20, warmup=5, only=None, table=CONFIGS):
    """Time every BASELINE config (or the one named `only`, else the ones
    whose name starts with it): mean µs over `steps` back-to-back calls (5x as many for
    HBM-bound configs, which take microseconds) after `warmup` calls and at
    least WARM_MS of untimed calls, with
    TFLOP/s, HBM GB/s and the fraction of the roofline that bounds the
    config.  HBM-bound configs rotate K/V sets (ROTATE_BYTES in total)."""
    from gqa_kernels.dispatch import _cu_count, choose_plan
    rows = []
    sel = table
    if only is not None:  # the config of that exact name, else those starting with it
        sel = [c for c in table if c[0] == only] or [c for c in table if c[0].startswith(only)]
    for name, b, hq, hkv, sq, skv, bound, d, *opt in sel:
        dtype_s = opt[0] if opt else "bf16"
        lse = bool(opt[1]) if len(opt) > 1 else False
        by1 = hbm_bytes(b, hq, hkv, sq, skv, d)
        nset = max(1, math.ceil(ROTATE_BYTES / by1)) if bound == "hbm" else 1
        q, kvs = _inputs(torch, b, hq, hkv, sq, skv, d, n_kv_sets=nset,
                         dtype=torch.float16 if dtype_s == "fp16" else torch.bfloat16)
        n = steps * 5 if bound == "hbm" else steps
        if lse:
            call = lambda i: gqa_flash_attn(q, *kvs[i % nset], causal=True, return_lse=True)  # noqa: E731
        else:
            call = lambda i: gqa_flash_attn(q, *kvs[i % nset], causal=True)  # noqa: E731
        ms = _time(torch, call, n, warmup, warm_ms=WARM_MS)
        fl = flops(b, hq, sq, skv, d)
        tflops, gbs = fl / (ms * 1e-3) / 1e12, by1 / (ms * 1e-3) / 1e9
        achieved, peak, unit = (tflops, PEAK_BF16_TFLOPS, "TFLOP/s") if bound == "mfma" else \
            (gbs, PEAK_HBM_GBS, "GB/s")
        route = choose_plan(b, hq, hkv, sq, skv, _cu_count(0), causal=True, head_dim=d)
        rows.append({"config": name, "B": b, "Hq": hq, "Hkv": hkv, "seq_q": sq, "seq_kv": skv, "D": d,
                     "dtype": dtype_s, "return_lse": lse, "us": ms * 1e3, "tflops": tflops, "gbs": gbs, "steps": n, "kv_sets": nset,
                     "route": route.kind + (f" splits={route.splits}" if route.kind in ("split", "chunks", "flat") else
                                            f" key-split blocks={route.fwd_split}" if route.fwd_split else ""),
                     "roofline": {"bound": bound, "achieved": achieved, "peak": peak, "unit": unit,
                                  "frac": achieved / peak, "flops_per_call": fl, "bytes_per_call": by1}})
        del q, kvs
        torch.cuda.empty_cache()
    return rows


if __name__ == "__main__":
    sys.exit(main())
