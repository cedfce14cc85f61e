#!/usr/bin/env python3
"""Headline benchmark of the fused GEMM + tile-publishing path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W]

A step is one pass of the hot path over one batch of synthetic input:
the bf16 shard GEMM A[8192,1024] x B[1024,8192] (one rank's K-shard of
K=8192) with 256x256 output tiles stored as bf16 into the fine-grained heap
and one uint32 ready flag published per tile.  Prints ONE JSON line.

The last line printed is the result: the GEMM's figures, and inside its
``roofline`` object also the reduce phase (``roofline.reduce``: the one-shot
reduce of 8 fp32 partial-C buffers [8192,8192] -> bf16, HBM-bound), the CPU
baseline of the same math on the host cores, and one-line summaries of the
other measurements.  Everything else (the cold-cache protocol run, the
library and matrix-core context figures, the other workloads) is printed
before it, one JSON line per group, each with a ``detail`` key, so that the
result line stays short.
"""

import argparse
import json
import math
import os
import statistics
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

PEAK_BF16_TFLOPS = 2500.0  # MI355X dense bf16 MFMA, published
PEAK_HBM_GBPS = 8000.0     # MI355X HBM3E, published

# HBM-side bytes per launch of the default kernels on this workload, from rocprofv3 --pmc FETCH_SIZE and
# WRITE_SIZE runs of this script, each scaled by what the same counter reads for the --copy-calibration
# kernel (profiles/gemm_all_scatter_bf16_8192x8192x1024.txt, profiles/one_shot_reduce_fp32x8_8192x8192.txt).
# Counters cannot be read from inside a run, so these are carried here and dropped for non-default variants.
GEMM_TRAFFIC_BYTES = 335108222
REDUCE_TRAFFIC_BYTES = 2281096192

M, N, K_SHARD, K_TOTAL = 8192, 8192, 1024, 8192
BLK_M, BLK_N, BLK_K, GSIZE_M, GRID = 256, 256, 64, 4, 256


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=500)
    ap.add_argument("--warmup", type=int, default=50)
    ap.add_argument("--settle-ms", type=float, default=300.0,
                    help="untimed launches of the same step before the warm-up, until this much time has passed: after "
                         "an idle period the GPU's power management first overshoots and then clamps the clocks for "
                         "~10 ms, which a short run would measure instead of the steady state")
    ap.add_argument("--variant", type=int, default=0, help="GEMM kernel tuning variant (0 = default)")
    ap.add_argument("--reduce-variant", type=int, default=0)
    ap.add_argument("--decoder-m", default="1,16,128,512,2048",
                    help="decoder workload: the row counts to run (comma-separated)")
    ap.add_argument("--gsize_m", type=int, default=GSIZE_M)
    ap.add_argument("--no-reduce", action="store_true", help="skip the reduce-phase measurement")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline")
    ap.add_argument("--no-coldcache", action="store_true", help="skip the cold-cache do_bench protocol run")
    ap.add_argument("--offheap-operands", action="store_true", help="keep A and B outside the fine-grained heap")
    ap.add_argument("--zero-operands", action="store_true",
                    help="all-zero A and B: nothing toggles in the matrix cores, the clocks stay up, and the time that "
                         "is left is the kernel's structure (not the metric's workload; the JSON line says so)")
    ap.add_argument("--decoder-split-k", type=int, default=0,
                    help="decoder workload: split_k of the two GEMMs (0: the launcher's choice, N > 1: N parts, "
                         "-1: stream-K)")
    ap.add_argument("--decoder-tiles", default="",
                    help="decoder workload: only this tile shape, as BLK_MxBLK_N (default: a sweep, and the "
                         "reference examples' default tile 256x64 beside it)")
    ap.add_argument("--shapes-gpus", default="1,2,4,8", help="shapes workload: the GPU counts the GEMMs are cut over")
    ap.add_argument("--shapes-partial", default="operand", choices=["operand", "fp32"],
                    help="shapes workload: element type of the one-shot producer's partial C: the operands' (what the "
                         "reference's 09 script allocates, benchmark.py:103,124) or fp32 (twice the bytes)")
    ap.add_argument("--shapes-algorithms", default="all_scatter,one_shot",
                    help="shapes workload: all_scatter (N-shards) and / or one_shot (K-shards, the producer)")
    ap.add_argument("--workload", choices=["headline", "atomic", "decoder", "shapes", "fused", "fp32"], default="headline",
                    help="headline: the 8192x8192x1024 shard GEMM + reduce (the metric's configuration); atomic: eight "
                         "K-shard GEMMs adding into one fp32 C; decoder: 6.7B-decoder-shaped shards for M in "
                         "{1,16,128,512,2048}; shapes: one rank's shard GEMM at every point of the reference's shape "
                         "sweep, beside the vendor library's; fused: the reference's one-shot program (store, signal, "
                         "wait, reduce, tile by tile) on two ranks resident side by side, against the producer + "
                         "reduce-kernel pair.  The last four print their own JSON line.")
    ap.add_argument("--no-other-workloads", action="store_true",
                    help="headline run: skip the atomic-accumulate and decoder-shard summaries")
    ap.add_argument("--no-context", action="store_true",
                    help="skip the two context figures: the library GEMM and the matrix cores' sustained rate")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="also launch a plain fp32 copy of [8192,8192] (256 MiB in, 256 MiB out): the kernel of known "
                         "size that scales the FETCH_SIZE / WRITE_SIZE counters of a rocprofv3 --pmc run")
    return ap.parse_args()


def timed_steps(fn, steps, warmup):
    """(wall seconds for `steps` calls, mean per-launch device ms).

    The device time comes from one pair of HIP events on the launch stream
    around the `steps` back-to-back launches: an event between every two
    launches would insert a ~11 us idle gap and a cache write-back before each
    kernel, which is not how the path runs.
    """
    import torch

    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    start.record()
    for _ in range(steps):
        fn()
    end.record()
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    return wall, start.elapsed_time(end) / steps


def cpu_baseline():
    """The oracle on the host cores at the full sizes of the two headline
    workloads: the shard GEMM (fp32 matmul + bf16 downcast of [8192,1024] x
    [1024,8192]) and the rank-ordered sum of eight fp32 [8192,8192] partials.
    About ten seconds in all."""
    import torch

    from oracle import iris_oracle as O

    g = torch.Generator().manual_seed(123)
    A = (torch.randn(M, K_SHARD, generator=g) * 0.02).to(torch.bfloat16)
    B = (torch.randn(N, K_SHARD, generator=g) * 0.02).to(torch.bfloat16).T
    O.shard_gemm(A, B, torch.bfloat16)  # warm-up
    times = []
    t_end = time.perf_counter() + 6.0
    while len(times) < 3 or (time.perf_counter() < t_end and len(times) < 20):
        t0 = time.perf_counter()
        O.shard_gemm(A, B, torch.bfloat16)
        times.append(time.perf_counter() - t0)
    med = statistics.median(times)
    del A, B
    # the reduce phase: 8 fp32 partials [8192, 8192] (2 GiB on the host) summed in rank order -> bf16
    parts = torch.empty(8, M, N)
    for r in range(8):
        parts[r].normal_(generator=g)
    O.one_shot_reduce(parts, torch.bfloat16)
    rtimes = []
    for _ in range(3):
        t0 = time.perf_counter()
        O.one_shot_reduce(parts, torch.bfloat16)
        rtimes.append(time.perf_counter() - t0)
    rmed = statistics.median(rtimes)
    return {
        "reduce_GBps": round((parts.numel() * 4 + M * N * 2) / rmed / 1e9, 2),
        "reduce_sample": "oracle one_shot_reduce of 8 fp32 partials [8192,8192] -> bf16 (the whole workload), 3 runs, "
                         "median",
        "value": 2.0 * M * N * K_SHARD / med / 1e12,
        "unit": "TFLOP/s",
        "cores": torch.get_num_threads(),
        "kind": "port",
        "sample": f"oracle shard_gemm (torch fp32 matmul + bf16 cast) on the whole A[8192,1024] x B[1024,8192], "
                  f"{len(times)} runs, median; os.cpu_count()={os.cpu_count()}",
    }


def steady_ms(fn, settle_s=0.2, n=200):
    """Mean device ms per call of `fn` over n back-to-back calls after a settle phase."""
    import torch

    t_end = time.perf_counter() + settle_s
    while time.perf_counter() < t_end:
        for _ in range(10):
            fn()
        torch.cuda.synchronize()
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    for _ in range(n):
        fn()
    e.record()
    torch.cuda.synchronize()
    return s.elapsed_time(e) / n


def shader_clock_mhz(fn, seconds=1.5):
    """Median shader clock, as ``rocm-smi --showclocks`` reports it, while ``fn`` runs back to back on the GPU
    (from a second thread; the first samples).  None where rocm-smi is missing or says nothing."""
    import re
    import subprocess
    import threading

    import torch

    # (not under a profiler: its preloaded tool library would start up inside every rocm-smi child as well)
    if "rocprofiler" in os.environ.get("LD_PRELOAD", "") or any(k.startswith(("ROCPROF", "ROCP_")) for k in os.environ):
        return None
    stop = threading.Event()

    def keep_busy():
        while not stop.is_set():
            for _ in range(100):
                fn()
            torch.cuda.synchronize()

    worker = threading.Thread(target=keep_busy)
    worker.start()
    samples = []
    try:
        time.sleep(0.5)  # (past the fast launches after an idle period)
        t_end = time.perf_counter() + seconds
        while time.perf_counter() < t_end:
            try:
                text = subprocess.run(["rocm-smi", "--showclocks"], capture_output=True, text=True, timeout=10).stdout
            except (OSError, subprocess.SubprocessError):
                break
            m = re.search(r"sclk clock level: \S+ \((\d+)Mhz\)", text)
            if m:
                samples.append(int(m.group(1)))
            time.sleep(0.1)
    finally:
        stop.set()
        worker.join()
    return int(statistics.median(samples)) if samples else None


def graph_ms(fn, per_graph=20, replays=20, settle_s=0.02, batches=3):
    """Mean device ms per call of `fn`, with `per_graph` calls captured in a HIP
    graph so that the host's launch cost (tens of microseconds per call through
    Python) does not bound what is measured.  The launchers only enqueue
    kernels on the current stream, so they can be captured.  Median of
    `batches` timed batches after a short settle phase."""
    import torch

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for _ in range(per_graph):
            fn()
    # Settle first: after an idle period the power management lets the first launches run fast and then clamps
    # the clocks for a few milliseconds, which a measurement of a few hundred microseconds would catch at random.
    t_end = time.perf_counter() + settle_s
    while time.perf_counter() < t_end:
        for _ in range(3):
            graph.replay()
        torch.cuda.synchronize()
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    times = []
    for _ in range(batches):
        s.record()
        for _ in range(replays):
            graph.replay()
        e.record()
        torch.cuda.synchronize()
        times.append(s.elapsed_time(e) / (per_graph * replays))
    return statistics.median(times)


def context_figures(a, b, c_global, flops, gemm_on):
    """Figures that put the headline number in context, measured the same
    way (settled clocks, back-to-back launches; ``gemm_on(a, b)`` launches the
    headline GEMM on other operands):

    * the vendor library's GEMM (torch.matmul -> hipBLASLt) on the same
      operands and output buffer, without flags;
    * what the matrix cores sustain with nothing but registers in the loop
      (``iris_mfma_probe_launch``), on operands drawn like the GEMM's and on
      zeros.  The board is power-limited: with operand bits that toggle, the
      sustained rate is well below the data-sheet peak, and no kernel on such
      data can exceed it.
    """
    import torch

    from iris_amd import ops, testing

    out = {}
    ms = steady_ms(lambda: torch.matmul(a, b, out=c_global))
    out["library_gemm"] = {"what": "torch.matmul (hipBLASLt) on the same operands, no tile flags",
                           "ms": round(ms, 5), "tflops": round(flops / (ms * 1e-3) / 1e12, 2)}
    # the same two kernels on all-zero operands of the same shape and strides: nothing toggles in the matrix
    # cores or on the way to them, the clocks stay up, and what is left is the kernels' structure
    az = torch.zeros((a.shape[0], a.stride(0)), dtype=a.dtype, device=a.device)[:, :a.shape[1]]
    bz = torch.zeros((b.shape[1], b.stride(1)), dtype=b.dtype, device=b.device)[:, :b.shape[0]].T
    ms = steady_ms(lambda: gemm_on(az, bz))
    out["gemm_on_zeros"] = {"what": "this kernel, all-zero operands", "ms": round(ms, 5),
                            "tflops": round(flops / (ms * 1e-3) / 1e12, 2)}
    ms = steady_ms(lambda: torch.matmul(az, bz, out=c_global))
    out["library_gemm_on_zeros"] = {"what": "torch.matmul (hipBLASLt), all-zero operands", "ms": round(ms, 5),
                                    "tflops": round(flops / (ms * 1e-3) / 1e12, 2)}
    # The shader clock under each of the four: on zeros nothing holds it back; on data the board's power cap
    # does, and the kernel that needs fewer clocks for the same work is held lower.
    out["shader_clock_mhz"] = {
        "how": "rocm-smi --showclocks sampled while the launch runs back to back, median",
        "gemm": shader_clock_mhz(lambda: gemm_on(a, b)),
        "library_gemm": shader_clock_mhz(lambda: torch.matmul(a, b, out=c_global)),
        "gemm_on_zeros": shader_clock_mhz(lambda: gemm_on(az, bz)),
        "library_gemm_on_zeros": shader_clock_mhz(lambda: torch.matmul(az, bz, out=c_global)),
    }
    del az, bz
    groups, iters = 256, 4000
    sink = torch.empty(groups * 512, dtype=torch.float32, device="cuda")
    for name, operands in (("random N(0,0.02)", (torch.randn(32768, device="cuda") * 0.02).to(torch.bfloat16)),
                           ("zeros", torch.zeros(32768, dtype=torch.bfloat16, device="cuda"))):
        fl = testing.mfma_probe(operands, sink, iters, groups)
        ms = steady_ms(lambda: testing.mfma_probe(operands, sink, iters, groups), n=100)
        out[f"mfma_sustained[{name}]"] = {"what": "register-only v_mfma_f32_16x16x32_bf16 loop, 8 waves per CU",
                                           "tflops": round(fl / (ms * 1e-3) / 1e12, 1)}
        # what the output stores of the headline launch cost next to the matrix cores, and whether spreading
        # them helps: 4 tiles a CU of register-only MFMAs (a 256x256x1024 tile's worth each) with 128 KiB of
        # write-through stores a tile, all at once / one KiB a wave and K-step / none (iris_store_probe_launch)
        tiles = 4
        region = torch.empty(tiles * groups * 131072, dtype=torch.uint8, device="cuda")
        t = {}
        for label, chunk in (("none", 0), ("tile_at_once", 16), ("one_store_per_k_step", 1)):
            t[label] = steady_ms(lambda: testing.store_probe(operands, sink, region, tiles, chunk, groups), n=100) * 1e3
        out[f"store_cost[{name}]"] = {
            "what": "register-only MFMAs of 4 tiles a CU + 128 MiB of write-through stores (16 one-KiB stores a wave "
                    "and tile), us per launch",
            "mfma_only_us": round(t["none"], 1),
            "tile_at_once_extra_us": round(t["tile_at_once"] - t["none"], 1),
            "one_store_per_k_step_extra_us": round(t["one_store_per_k_step"] - t["none"], 1)}
        del region
    return out


def run_fp32(args, emit=True):
    """The headline shard with fp32 operands (the reference scripts' --datatype fp32): A[8192,1024] x B[1024,8192]
    on K-shard views, fp32 C behind a flag per 256 x 256 tile, beside the vendor library's fp32 GEMM on the same
    operands.  The matrix cores run fp32 at 157.3 TFLOP/s."""
    import torch

    import iris_amd
    from iris_amd import ops

    M = N = 8192
    K, K_total = 1024, 8192
    shmem = iris_amd.iris(2 << 30)
    a_full = shmem.zeros((M, K_total), dtype=torch.float32)
    bt_full = shmem.zeros((N, K_total), dtype=torch.float32)
    a_full.normal_(0, 0.02)
    bt_full.normal_(0, 0.02)
    a, b = a_full[:, :K], bt_full[:, :K].T
    cg = shmem.zeros((M, N), dtype=torch.float32)
    flags = shmem.zeros((1024,), dtype=torch.int32)
    lib = torch.empty((M, N), dtype=torch.float32, device="cuda")
    largs = (a, b, None, cg, flags, None, 0, 1, 256, 256, 256, 64, 4, ops.EPI_ALL_SCATTER)
    kw = dict(num_xcds=ops.default_num_xcds(shmem.get_cu_count(), 256))

    def ours():
        ops.gemm_launch(*largs, **kw)

    def library():
        torch.matmul(a, b, out=lib)

    ours()
    library()
    torch.cuda.synchronize()
    err = (cg - lib).abs().max().item()
    assert err <= 1e-4 * lib.abs().max().item(), f"fp32 GEMM differs from the library's by {err}"
    assert flags.cpu().tolist() == [1] * 1024
    flops = 2.0 * M * N * K
    ms = steady_ms(ours, n=50)
    lib_ms = steady_ms(library, n=50)
    peak = 157.3
    result = {
        "metric": "shard GEMM + flag-published epilogue with fp32 operands", "value": round(flops / ms / 1e9, 2),
        "unit": "TFLOP/s", "n_gpus": 1, "ms_per_step": round(ms, 5), "higher_is_better": True, "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": "fp32 A[8192,1024] x B[1024,8192] (K-shard views, lda=ldb=8192), 256x256 tiles -> fp32 "
                               "in the fine-grained heap, one ready flag per tile", "grid": 256},
        "kernel": ops.gemm_plan_name(*largs, **kw),
        "roofline": {"bound": "mfma", "achieved": round(flops / ms / 1e9, 2), "peak": peak, "unit": "TFLOP/s",
                     "frac": round(flops / ms / 1e9 / peak, 4), "traffic": None},
        "library_ms": round(lib_ms, 5), "library_tflops": round(flops / lib_ms / 1e9, 2),
        "max_abs_diff_vs_library": err,
    }
    if emit:
        print(json.dumps(result))
    return result


def run_atomic(args, emit=True):
    """eight sequential bf16 K-shard GEMMs A_i[4096,512] x
    B_i[512,4096], each adding its tiles with fp32 atomics into one C[4096,4096]
    in the heap."""
    import torch

    import iris_amd
    from iris_amd import ops

    Ma = Na = 4096
    ks, shards = 512, 8
    shmem = iris_amd.iris(1 << 29)
    g = torch.Generator().manual_seed(123)
    A = (torch.randn(Ma, ks * shards, generator=g) * 0.05).to(torch.bfloat16)
    B = (torch.randn(Na, ks * shards, generator=g) * 0.05).to(torch.bfloat16)
    a_full = shmem.zeros((Ma, ks * shards), dtype=torch.bfloat16)
    a_full.copy_(A)
    bt_full = shmem.zeros((Na, ks * shards), dtype=torch.bfloat16)
    bt_full.copy_(B)
    c = shmem.zeros((Ma, Na), dtype=torch.float32)
    hb = shmem.get_heap_bases()
    blk_m, blk_n, grid = 256, 256, 256
    num_xcds = ops.default_num_xcds(shmem.get_cu_count(), grid)

    def step():
        for i in range(shards):
            ops.gemm_launch(a_full[:, i * ks:(i + 1) * ks], bt_full[:, i * ks:(i + 1) * ks].T, None, c, None, hb, 0, 1,
                            grid, blk_m, blk_n, 64, 6, ops.EPI_ATOMIC_ADD, num_xcds=num_xcds, variant=args.variant)

    step()
    torch.cuda.synchronize()
    ref = torch.matmul(a_full.float(), bt_full.float().T)
    err = (c - ref).abs().max().item()
    assert torch.allclose(c, ref, rtol=1e-2, atol=1e-2), f"atomic accumulate differs from the fp32 product: {err}"
    ms = steady_ms(step, n=max(10, args.steps // 10))
    flops = 2.0 * Ma * Na * ks * shards
    updates = Ma * Na * shards
    # what the chip takes when it does nothing else: one coalesced fp32 atomic add per element of the same C,
    # eight passes (the kernel of the reference's atomic_add microbenchmark, examples/04_atomic_add)
    def atomics_only():
        for _ in range(shards):
            ops.p2p_bench("atomic_add", c.view(-1), None, hb, 0, 0, 1, block_size=512)

    ceil_ms = steady_ms(atomics_only, n=max(10, args.steps // 10))
    result = {
        "metric": "atomic-accumulate epilogue: 8 K-shard GEMMs into one fp32 C", "value": round(flops / ms / 1e9, 2),
        "unit": "TFLOP/s", "n_gpus": 1, "ms_per_step": round(ms, 5), "higher_is_better": True, "dtype": "bf16",
        "data": "synthetic",
        "config": {"workload": "8 sequential bf16 GEMMs A_i[4096,512] x B_i[512,4096] with fp32 atomicAdd of 256x256 "
                               "tiles into C[4096,4096] in the fine-grained heap", "grid": grid},
        "atomic_updates_per_s": round(updates / (ms * 1e-3), 0),
        "atomic_GBps_at_4B": round(updates * 4 / (ms * 1e-3) / 1e9, 1),
        "atomic_ceiling": {"what": "the same 8 x 16.8 M fp32 atomic adds on C with no GEMM in front "
                                   "(iris_p2p_bench_launch, ATOMIC_ADD)",
                           "ms": round(ceil_ms, 5), "updates_per_s": round(updates / (ceil_ms * 1e-3), 0),
                           "frac_of_ceiling": round(ceil_ms / ms, 4)},
        "max_abs_err_vs_fp32": err,
    }
    if emit:
        print(json.dumps(result))
    return result


def side_by_side_streams(shmem):
    """Two streams of this process that really run side by side on the device.
    HIP maps streams onto a few hardware queues and two streams on one queue run
    one after the other, so candidate pairs are probed with the flag protocol
    itself: a one-tile consumer with a bounded wait (20 ms) on one stream, then
    the signal it waits for on the other."""
    import torch

    from iris_amd import ops

    off = shmem.heap_offset
    ws = shmem.get_num_ranks()
    c = shmem.zeros((64, 64), dtype=torch.float32)
    cg = shmem.zeros((64, 64), dtype=torch.float32)
    flag = shmem.zeros((1,), dtype=torch.int32)
    hb = shmem.get_heap_bases()
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    streams = [torch.cuda.Stream() for _ in range(4)]
    for st in streams:  # the first submission to a new stream takes milliseconds
        with torch.cuda.stream(st):
            torch.zeros(8, device="cuda").add_(1)
    torch.cuda.synchronize()
    try:
        for sb in streams:
            for sa in streams:
                if sa is sb:
                    continue
                for r in range(ws):
                    shmem.on_rank(flag, r).zero_()
                status.zero_()
                torch.cuda.synchronize()
                with torch.cuda.stream(sb):
                    ops.one_shot_reduce(c, cg, flag, hb, 0, 2, 64, 64, 1, num_sms=1, variant=8, status=status,
                                        spin_timeout_ticks=2_000_000)
                with torch.cuda.stream(sa):
                    ops.signal_tiles(shmem.on_rank(flag, 1), hb, 1, 1, 2)
                torch.cuda.synchronize()
                if int(status.item()) == 0:
                    return sa, sb
    finally:
        shmem.heap_offset = off
    raise RuntimeError("no two streams of this process run side by side on the device")


def run_fused(args, emit=True):
    """The reference's 09 program as it runs (gemm_one_shot_all_reduce.py:197-271):
    every program stores its partial tile, signals the other rank, waits for
    the tile's flag on its own rank, sums the tile over the ranks and stores
    it, tile by tile.  Two ranks of 128 programs each, resident side by side
    on the one GPU (one stream per rank), each computing
    [8192, 1024] x [1024, 8192] of a K = 2048 product into fp32 partials and a
    bf16 result; against the same work as two kernels per rank on one stream
    (producer GEMM on 256 programs, then the reduce kernel)."""
    import torch

    import iris_amd
    from iris_amd import ops
    from oracle import iris_oracle as O

    ws, ks = 2, K_SHARD
    blk_m, blk_n, gsize = 256, 256, 6  # the 09 script's own tile and group size
    half_second = 50_000_000            # every wait is bounded: 0.5 s of the 100 MHz wall clock
    shmem = iris_amd.iris(1 << 30, virtual_ranks=ws)
    on = shmem.on_rank
    dtype = torch.bfloat16
    g = torch.Generator().manual_seed(123)
    A = (torch.randn(M, ks * ws, generator=g) * 0.02).to(dtype)
    B = (torch.randn(N, ks * ws, generator=g) * 0.02).to(dtype)
    a_full = shmem.zeros((M, ks * ws), dtype=dtype)
    a_full.copy_(A)
    bt_full = shmem.zeros((N, ks * ws), dtype=dtype)
    bt_full.copy_(B)
    del A, B
    c = shmem.zeros((M, N), dtype=torch.float32)
    cg = shmem.zeros((M, N), dtype=dtype)
    total = ops.cdiv(M, blk_m) * ops.cdiv(N, blk_n)
    flags = shmem.zeros((total,), dtype=torch.int32)
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    hb = shmem.get_heap_bases()
    xcds = ops.default_num_xcds(shmem.get_cu_count(), 128)
    sa, sb = side_by_side_streams(shmem)

    def clear():
        for r in range(ws):
            for t in (c, cg, flags):
                on(t, r).zero_()
        status.zero_()

    def launch(r, phase, grid):
        ops.gemm_launch(a_full[:, r * ks:(r + 1) * ks], bt_full[:, r * ks:(r + 1) * ks].T, on(c, r), on(cg, r),
                        on(flags, r), hb, r, ws, grid, blk_m, blk_n, 64, gsize, ops.EPI_ONE_SHOT, phase=phase,
                        num_xcds=xcds, status=status, spin_timeout_ticks=half_second)

    def in_program():  # both ranks' programs on the device together
        for r, st in enumerate((sa, sb)):
            with torch.cuda.stream(st):
                launch(r, ops.PHASE_FUSED, 128)

    def two_kernels():  # both producers, then both reduce kernels, on one stream
        for r in range(ws):
            launch(r, ops.PHASE_PRODUCE, 256)
        for r in range(ws):
            ops.one_shot_reduce(on(c, r), on(cg, r), on(flags, r), hb, r, ws, blk_m, blk_n, gsize, num_xcds=xcds,
                                status=status, spin_timeout_ticks=half_second)

    # correctness first, on the whole matrices: the partials against each other's builds, and the result of both
    # forms bit for bit against the oracle's rank-ordered sum of those partials
    results = {}
    for name, run in (("in_program", in_program), ("two_kernels", two_kernels)):
        clear()
        torch.cuda.synchronize()
        run()
        torch.cuda.synchronize()
        assert int(status.item()) == 0, f"{name}: a flag wait timed out"
        partials = torch.stack([on(c, r).cpu() for r in range(ws)])
        want = O.one_shot_reduce(partials, dtype)
        for r in range(ws):
            assert torch.equal(on(cg, r).cpu(), want), f"{name}: rank {r} is not the rank-ordered sum of the partials"
            assert int(on(flags, r).abs().max().item()) == 0, f"{name}: flags of rank {r} not consumed"
        results[name] = partials
    assert torch.equal(results["in_program"], results["two_kernels"]), "the two forms computed different partials"
    del results, partials, want

    steps = max(5, min(args.steps, 100))
    start, end_a, end_b = (torch.cuda.Event(enable_timing=True) for _ in range(3))

    def timed_in_program():
        ms = []
        for _ in range(steps):
            torch.cuda.synchronize()
            with torch.cuda.stream(sa):
                start.record()
            sb.wait_event(start)
            in_program()
            with torch.cuda.stream(sa):
                end_a.record()
            with torch.cuda.stream(sb):
                end_b.record()
            torch.cuda.synchronize()
            ms.append(max(start.elapsed_time(end_a), start.elapsed_time(end_b)))
        return ms

    def timed_two_kernels():
        ms = []
        for _ in range(steps):
            torch.cuda.synchronize()
            start.record()
            two_kernels()
            end_a.record()
            torch.cuda.synchronize()
            ms.append(start.elapsed_time(end_a))
        return ms

    # settle the clocks on this work, then alternate the two forms
    t_end = time.perf_counter() + args.settle_ms * 1e-3
    while time.perf_counter() < t_end:
        two_kernels()
        torch.cuda.synchronize()
    timed_in_program()
    t_in, t_two = timed_in_program(), timed_two_kernels()
    assert int(status.item()) == 0, "a flag wait timed out during the timed runs"
    for r in range(ws):
        assert int(on(flags, r).abs().max().item()) == 0
    ms_in, ms_two = statistics.median(t_in), statistics.median(t_two)
    flops = ws * 2.0 * M * N * ks
    rbytes = ws * (ws * M * N * 4 + M * N * 2)
    out = {
        "metric": "one-shot all-reduce GEMM as the reference program runs it (store, signal, wait, reduce per tile), "
                  "two ranks side by side on one GPU",
        "value": round(flops / (ms_in * 1e-3) / 1e12, 2), "unit": "TFLOP/s", "n_gpus": 1, "steps": steps,
        "ms_per_step": round(ms_in, 5), "higher_is_better": True, "dtype": "bf16", "data": "synthetic",
        "config": {"workload": "2 ranks x 128 programs of IRIS_PHASE_FUSED, each [8192,1024] x [1024,8192] (K-shard views "
                               "of K = 2048), 256x256 tiles, fp32 partials, bf16 result on both ranks; one stream per rank",
                   "ranks": ws, "programs_per_rank": 128, "BLK_M": blk_m, "BLK_N": blk_n, "gsize_m": gsize},
        "in_program": {"ms": round(ms_in, 5), "min_ms": round(min(t_in), 5), "max_ms": round(max(t_in), 5),
                       "tflops": round(flops / (ms_in * 1e-3) / 1e12, 2)},
        "two_kernels": {"what": "the same work as kernels on one stream: both ranks' producer GEMMs (256 programs), then "
                                "both ranks' reduce kernels", "ms": round(ms_two, 5), "min_ms": round(min(t_two), 5),
                        "max_ms": round(max(t_two), 5), "tflops": round(flops / (ms_two * 1e-3) / 1e12, 2)},
        "in_program_vs_two_kernels": round(ms_two / ms_in, 3),
        "reduce_bytes": rbytes,
        "checked": "both forms bit-exact against the oracle's rank-ordered sum of the partials on the whole "
                   "[8192,8192], flags back to 0, status 0",
    }
    if emit:
        print(json.dumps(out))
    del shmem
    return out



# The reference's shape sweep (examples/benchmark/bench_all_shapes.py:103-187): the six GEMMs of
# dataset/mini.json (m = 8192), each cut over 1, 2, 4 and 8 GPUs, with the tile and group size that
# dataset/tiling.json holds for the rank's shard shape: (m, k, n / gpus) for the all-scatter, (m, k / gpus, n) for
# the reduce algorithms.  (n, k) -> gpus -> ((BLK_M, BLK_N, gsize_m) all-scatter, (...) one-shot), as looked up there.
SWEEP_SHAPES = {
    (4096, 12288): {1: ((128, 128, 6), (128, 128, 6)), 2: ((256, 256, 6), (128, 128, 6)),
                    4: ((128, 256, 6), (256, 256, 2)), 8: ((128, 128, 6), (256, 256, 2))},
    (4096, 14336): {1: ((128, 128, 6), (128, 128, 6)), 2: ((256, 256, 6), (128, 128, 6)),
                    4: ((128, 256, 6), (256, 256, 2)), 8: ((128, 128, 6), (256, 256, 2))},
    (3584, 14336): {1: ((128, 256, 6), (128, 256, 6)), 2: ((128, 128, 2), (128, 256, 6)),
                    4: ((256, 128, 1), (128, 256, 6)), 8: ((256, 64, 1), (128, 256, 6))},
    (4608, 36864): {1: ((256, 256, 2), (256, 256, 2)), 2: ((256, 256, 6), (256, 256, 2)),
                    4: ((256, 128, 1), (256, 256, 2)), 8: ((256, 64, 1), (256, 256, 2))},
    (8192, 28672): {1: ((128, 256, 6), (128, 256, 6)), 2: ((128, 128, 6), (128, 256, 6)),
                    4: ((256, 256, 6), (128, 256, 6)), 8: ((128, 256, 6), (128, 256, 6))},
    (8192, 30720): {1: ((128, 256, 6), (128, 256, 6)), 2: ((128, 128, 6), (128, 256, 6)),
                    4: ((256, 256, 6), (128, 256, 6)), 8: ((128, 256, 6), (128, 256, 6))},
}


def sweep_tile(blk_m, blk_n):
    """The tile the sweep launches for a tile of the table: it runs 128 x 256 and 128 x 128 entries as 256 x 128
    (bench_all_shapes.py:161-166)."""
    return (256, 128) if (blk_m, blk_n) in ((128, 256), (128, 128)) else (blk_m, blk_n)


def run_shapes(args, emit=True):
    """One rank's shard GEMM for every point of the reference's shape sweep, at the sweep's tile, beside the vendor
    library's plain GEMM on the same shard: the all-scatter ([8192, k] x [k, n / gpus], the tile stored into
    every rank's C behind its flag) and the producer of the one-shot all-reduce ([8192, k / gpus] x [k / gpus, n]
    on K-shard views of the whole operands, a partial C of the operands' type behind flags on the other ranks, as
    the reference's 09 script allocates it, benchmark.py:103,124; --shapes-partial fp32 for fp32 partials)."""
    import torch

    import iris_amd
    from iris_amd import ops

    m = 8192
    gpus_list = [int(v) for v in args.shapes_gpus.split(",")]
    points = []
    for ws in gpus_list:
        # per rank: A and B of the largest shape (0.6 + 0.5 GB), bf16 C, the partial, flags
        shmem = iris_amd.iris(2 << 30, virtual_ranks=ws)
        hb = shmem.get_heap_bases()
        xcds = ops.default_num_xcds(shmem.get_cu_count(), 256)
        rank = ws - 1
        for (n, k), by_gpus in SWEEP_SHAPES.items():
            if ws not in by_gpus:
                continue
            off = shmem.heap_offset
            a = shmem.zeros((m, k), dtype=torch.bfloat16)
            bt = shmem.zeros((n, k), dtype=torch.bfloat16)  # B = bt.T: K-contiguous, as the scripts pass it
            a.normal_(0, 0.02)
            bt.normal_(0, 0.02)
            cg = shmem.zeros((m, n), dtype=torch.bfloat16)
            part = shmem.zeros((m, n), dtype=torch.float32 if args.shapes_partial == "fp32" else torch.bfloat16)
            ns, ks = n // ws, k // ws
            for algorithm, (bm0, bn0, gsize_m) in zip(("all_scatter", "one_shot"), by_gpus[ws]):
                if algorithm not in args.shapes_algorithms.split(","):
                    continue
                bm, bn = sweep_tile(bm0, bn0)
                if algorithm == "all_scatter":
                    a_r, b_r, n_r = a, bt[rank * ns:(rank + 1) * ns].T, ns
                else:
                    a_r, b_r, n_r = a[:, rank * ks:(rank + 1) * ks], bt[:, rank * ks:(rank + 1) * ks].T, n
                flags = shmem.zeros((ops.cdiv(m, bm) * ops.cdiv(n_r, bn),), dtype=torch.int32)
                # the wrappers' P / locks buffers (benchmark.py:136-142): with them the launcher may split K
                P = shmem.zeros((256, bm * bn), dtype=torch.float32)
                locks = shmem.zeros((256,), dtype=torch.int32)
                if algorithm == "all_scatter":
                    largs = (a_r, b_r, None, shmem.on_rank(cg, rank), shmem.on_rank(flags, rank), hb, rank, ws, 256,
                             bm, bn, 64, gsize_m, ops.EPI_ALL_SCATTER)
                    kw = dict(num_xcds=xcds, partials=P, locks=locks)
                    got = lambda: shmem.on_rank(cg, 0)[:, rank * ns:(rank + 1) * ns]
                else:
                    largs = (a_r, b_r, shmem.on_rank(part, rank), shmem.on_rank(cg, rank),
                             shmem.on_rank(flags, rank), hb, rank, ws, 256, bm, bn, 64, gsize_m, ops.EPI_ONE_SHOT)
                    kw = dict(num_xcds=xcds, phase=ops.PHASE_PRODUCE, partials=P, locks=locks)
                    got = lambda: shmem.on_rank(part, rank)
                lib = torch.empty((m, n_r), dtype=torch.bfloat16, device="cuda")

                def ours():
                    ops.gemm_launch(*largs, **kw)

                def library():
                    torch.matmul(a_r, b_r, out=lib)

                ours()
                library()
                torch.cuda.synchronize()
                # the library's result is bf16 and sums in another order: agreement to two bf16 roundings
                diff = (got().float() - lib.float()).abs().max().item()
                scale = lib.float().abs().max().item()
                assert diff <= 2e-2 * scale, f"{algorithm} n={n} k={k} gpus={ws}: differs from the library's by {diff}"
                tiles_done = int((shmem.on_rank(flags, 0) > 0).sum().item())
                assert tiles_done == (flags.numel() if ws > 1 or algorithm == "all_scatter" else 0)
                flops = 2.0 * m * n_r * a_r.shape[1]
                t = {}
                for name, fn in (("ours", ours), ("library", library)):
                    est = steady_ms(fn, settle_s=0.05, n=3)
                    t[name] = steady_ms(fn, settle_s=0.1, n=max(5, min(200, int(150.0 / est))))
                points.append({
                    "n": n, "k": k, "gpus": ws, "algorithm": algorithm, "shard": [m, n_r, a_r.shape[1]],
                    "tile": [bm, bn], "gsize_m": gsize_m, "kernel": ops.gemm_plan_name(*largs, **kw),
                    "split_k": ops.gemm_split_k(*largs, **kw),
                    "us": round(t["ours"] * 1e3, 1), "tflops": round(flops / t["ours"] / 1e9, 1),
                    "library_us": round(t["library"] * 1e3, 1), "library_tflops": round(flops / t["library"] / 1e9, 1),
                    "vs_library": round(t["library"] / t["ours"], 3)})
                del lib
            shmem.heap_offset = off
        del shmem
    ratios = sorted(p["vs_library"] for p in points)
    out = {
        "metric": "shard GEMM + tile-publishing epilogue over the reference's shape sweep: rate against the vendor "
                  "library's plain GEMM on the same shard (geometric mean)",
        "value": round(math.exp(sum(math.log(r) for r in ratios) / len(ratios)), 3), "unit": "x",
        "n_gpus": 1, "higher_is_better": True, "dtype": "bf16", "data": "synthetic",
        "config": {"workload": "dataset/mini.json's six GEMMs (m = 8192) cut over " + args.shapes_gpus + " GPUs at the "
                               "tiles of dataset/tiling.json, one rank's share on one GPU with the other ranks' "
                               "heaps in the same HBM",
                   "one_shot_partial": "fp32" if args.shapes_partial == "fp32" else "bf16 (the operands' type)"},
        "worst": ratios[0], "best": ratios[-1], "points": points}
    if emit:
        print(json.dumps(out))
    return out


def run_decoder(args, emit=True):
    """6.7B-decoder-shaped shards (hidden 4096, FFN 11008,
    1/8 shard = 1376).  Gate/up: [M,4096] x [4096,1376] scattered into every
    rank's [M, 8*1376] at column rank*1376; down: [M,1376] x [1376,4096] as a
    partial, then the one-shot reduce of the 8 ranks' partials."""
    import torch

    import iris_amd
    from iris_amd import ops

    ws, hidden, ffn = 8, 4096, 1376
    shmem = iris_amd.iris(1 << 28, virtual_ranks=ws)
    hb = shmem.get_heap_bases()
    g = torch.Generator().manual_seed(123)
    rows = []
    # the kernel builds by name: a four-wave tile comes with fetching waves ("_f4") and plain
    variants, v = {}, 1
    while (vname := ops.gemm_variant_name(torch.bfloat16, False, False, v)) is not None:
        variants.setdefault(vname, v)
        v += 1

    def plain_build_of(kernel):
        """Variant number of the build of `kernel`'s tile shape and wave layout in which every wave fetches its
        share of the operands, or None if `kernel` is such a build already (or is run in parts of the caller's tiles,
        which a launch that names a variant is not)."""
        base = kernel.split("+")[0]
        if not base.endswith("_f4") or "+parts_of_tiles" in kernel:
            return None
        shape, waves = base.split("x")[:2], base.split("_")[1]
        for cand, num in variants.items():
            if not cand.endswith("_f4") and cand.split("x")[:2] == shape and cand.split("_")[1] == waves:
                return num
        return None
    for Mt in [int(t) for t in args.decoder_m.split(",")]:
        off = shmem.heap_offset
        x = shmem.zeros((Mt, hidden), dtype=torch.bfloat16)
        x.copy_((torch.randn(Mt, hidden, generator=g) * 0.02).to(torch.bfloat16))
        wg = shmem.zeros((ffn, hidden), dtype=torch.bfloat16)
        wg.copy_((torch.randn(ffn, hidden, generator=g) * 0.02).to(torch.bfloat16))
        wd = shmem.zeros((hidden, ffn), dtype=torch.bfloat16)
        wd.copy_((torch.randn(hidden, ffn, generator=g) * 0.02).to(torch.bfloat16))
        h = shmem.zeros((Mt, ffn), dtype=torch.bfloat16)
        h.copy_((torch.randn(Mt, ffn, generator=g) * 0.02).to(torch.bfloat16))
        gate_all = shmem.zeros((Mt, ws * ffn), dtype=torch.bfloat16)
        part = shmem.zeros((Mt, hidden), dtype=torch.float32)
        out = shmem.zeros((Mt, hidden), dtype=torch.bfloat16)
        rank = 3
        ref_up = torch.matmul(x.float(), wg.float().T)
        ref_dn = torch.matmul(h.float(), wd.float().T)
        lib_up = torch.empty((Mt, ffn), dtype=torch.bfloat16, device="cuda")
        lib_dn = torch.empty((Mt, hidden), dtype=torch.bfloat16, device="cuda")
        # the caller owns the tile shape (BLK_M, BLK_N); sweep the shapes a caller would consider and keep
        # the fastest for each GEMM
        shapes = [(bm, bn) for bm in (64, 128, 256) for bn in (64, 128, 256) if bm <= max(64, 2 * Mt)]
        ref_tile = (256, 64)  # BLK_M x BLK_N the reference's 07 and 09 scripts default to (benchmark.py:40-41)
        if args.decoder_tiles:
            shapes = [tuple(int(v) for v in args.decoder_tiles.lower().split("x"))]
        elif ref_tile not in shapes:
            shapes.append(ref_tile)
        best, at_ref, plain_at = {}, {}, {}
        for bm, bn in shapes:
            t_up = ops.cdiv(Mt, bm) * ops.cdiv(ffn, bn)
            t_dn = ops.cdiv(Mt, bm) * ops.cdiv(hidden, bn)
            hoff = shmem.heap_offset
            flags_up = shmem.zeros((t_up,), dtype=torch.int32)
            flags_dn = shmem.zeros((t_dn,), dtype=torch.int32)
            grid_up = grid_dn = 256
            xcds = ops.default_num_xcds(shmem.get_cu_count(), 256)  # what the matmul wrappers pass
            # the wrappers' P / locks buffers: with them the launcher may split K over idle programs
            P = shmem.zeros((256, bm * bn), dtype=torch.float32)
            locks = shmem.zeros((256,), dtype=torch.int32)

            def up():
                ops.gemm_launch(x, wg.T, None, shmem.on_rank(gate_all, rank), shmem.on_rank(flags_up, rank), hb, rank,
                                ws, grid_up, bm, bn, 64, 4, ops.EPI_ALL_SCATTER, notify=True, partials=P, locks=locks,
                                num_xcds=xcds, split_k=args.decoder_split_k)

            def up_plain_build():  # gate/up through the build without fetching waves
                ops.gemm_launch(x, wg.T, None, shmem.on_rank(gate_all, rank), shmem.on_rank(flags_up, rank), hb, rank,
                                ws, grid_up, bm, bn, 64, 4, ops.EPI_ALL_SCATTER, notify=True, partials=P, locks=locks,
                                num_xcds=xcds, variant=plain_variant, split_k=args.decoder_split_k)

            def up_one():  # the same GEMM with the launching rank as its only destination (a plain GEMM + flags)
                ops.gemm_launch(x, wg.T, None, shmem.on_rank(gate_all, rank), shmem.on_rank(flags_up, rank), hb[rank:],
                                0, 1, grid_up, bm, bn, 64, 4, ops.EPI_ALL_SCATTER, notify=True, partials=P, locks=locks,
                                num_xcds=xcds, split_k=args.decoder_split_k)

            def down():
                ops.gemm_launch(h, wd.T, shmem.on_rank(part, rank), shmem.on_rank(out, rank),
                                shmem.on_rank(flags_dn, rank), hb, rank, ws, grid_dn, bm, bn, 64, 6,
                                ops.EPI_ONE_SHOT, phase=ops.PHASE_PRODUCE, partials=P, locks=locks, num_xcds=xcds,
                                split_k=args.decoder_split_k)

            def reduce():
                ops.one_shot_reduce(shmem.on_rank(part, rank), shmem.on_rank(out, rank),
                                    shmem.on_rank(flags_dn, rank), hb, rank, ws, bm, bn, 6, wait_flags=False)

            shmem.on_rank(gate_all, 5).zero_()
            shmem.on_rank(part, rank).zero_()
            up()
            down()
            torch.cuda.synchronize()
            got = shmem.on_rank(gate_all, 5)[:, rank * ffn:(rank + 1) * ffn].float()
            assert torch.allclose(got, ref_up, rtol=1e-2, atol=1e-2), "gate/up scatter differs from the fp32 product"
            assert torch.allclose(shmem.on_rank(part, rank), ref_dn, rtol=1e-2, atol=1e-2), "down partial differs"
            up_args = (x, wg.T, None, shmem.on_rank(gate_all, rank), shmem.on_rank(flags_up, rank), hb, rank, ws,
                       grid_up, bm, bn, 64, 4, ops.EPI_ALL_SCATTER)
            dn_args = (h, wd.T, shmem.on_rank(part, rank), shmem.on_rank(out, rank), shmem.on_rank(flags_dn, rank),
                       hb, rank, ws, grid_dn, bm, bn, 64, 6, ops.EPI_ONE_SHOT)
            plan_kw = dict(partials=P, locks=locks, num_xcds=xcds, split_k=args.decoder_split_k)
            sk = {"gate_up": ops.gemm_split_k(*up_args, **plan_kw),
                  "down": ops.gemm_split_k(*dn_args, phase=ops.PHASE_PRODUCE, **plan_kw), "reduce": 1}
            kern = {"gate_up": ops.gemm_plan_name(*up_args, **plan_kw),
                    "down": ops.gemm_plan_name(*dn_args, phase=ops.PHASE_PRODUCE, **plan_kw), "reduce": "reduce"}
            plain_variant = plain_build_of(kern["gate_up"])
            runs = [("gate_up", up), ("down", down), ("reduce", reduce), ("gate_up_one", up_one)]
            if plain_variant is not None:
                runs.append(("gate_up_plain", up_plain_build))
            for name, fn in runs:
                if name in ("gate_up_one", "gate_up_plain"):
                    kern[name], sk[name] = kern["gate_up"], sk["gate_up"]
                ms = graph_ms(fn, 10, 10)
                if name == "gate_up_plain":  # kept for the tile that wins the sweep, not a candidate itself
                    plain_at[(bm, bn)] = ms
                    continue
                if (bm, bn) == ref_tile:
                    at_ref[name] = (ms, kern[name], sk[name])
                    if not args.decoder_tiles and bm > max(64, 2 * Mt):
                        continue  # taller than a caller would pick for this M: reported, not part of the sweep
                if name not in best or ms < best[name][0]:
                    best[name] = (ms, [bm, bn], sk[name], kern[name])
            shmem.heap_offset = hoff
        ms_up, ms_dn, ms_red = best["gate_up"][0], best["down"][0], best["reduce"][0]
        fl = 2.0 * Mt * hidden * ffn
        wbytes = hidden * ffn * 2
        rows.append({
            "M": Mt, "tile_up": best["gate_up"][1], "tile_down": best["down"][1], "tile_reduce": best["reduce"][1],
            "split_k_up": best["gate_up"][2], "split_k_down": best["down"][2],
            "kernel_up": best["gate_up"][3], "kernel_down": best["down"][3],
            "gate_up_us": round(ms_up * 1e3, 2), "gate_up_tflops": round(fl / ms_up / 1e9, 2),
            "gate_up_weight_GBps": round(wbytes / ms_up / 1e6, 1),
            "down_us": round(ms_dn * 1e3, 2), "down_tflops": round(fl / ms_dn / 1e9, 2),
            "down_weight_GBps": round(wbytes / ms_dn / 1e6, 1),
            "reduce_us": round(ms_red * 1e3, 2),
            "reduce_GBps": round((ws * Mt * hidden * 4 + Mt * hidden * 2) / ms_red / 1e6, 1),
            # the same three launches with the tile the reference's scripts default to, no sweep
            "at_reference_default_tile_256x64": {k: {"us": round(v[0] * 1e3, 2), "kernel": v[1], "split_k": v[2]}
                                                 for k, v in at_ref.items()},
            # gate/up with one destination instead of eight: what the library's figure below compares with like for
            # like (the scatter writes 8 x the output: 45 MB at 2048 rows, ~7 us at the rate HBM takes stores)
            "gate_up_one_destination_us": round(best["gate_up_one"][0] * 1e3, 2),
            # gate/up at the winning tile through the build in which every wave fetches its own share of the
            # operands (no fetching waves); null where the winning kernel is such a build
            "gate_up_without_fetching_waves_us": (round(plain_at[tuple(best["gate_up"][1])] * 1e3, 2)
                                                  if tuple(best["gate_up"][1]) in plain_at else None),
            # the vendor library's plain GEMM on the same operands (one destination, no flags), same timing
            "library_gate_up_us": round(graph_ms(lambda: torch.matmul(x, wg.T, out=lib_up), 10, 10) * 1e3, 2),
            "library_down_us": round(graph_ms(lambda: torch.matmul(h, wd.T, out=lib_dn), 10, 10) * 1e3, 2),
        })
        shmem.heap_offset = off  # the next M reuses the heap
    big = rows[-1]
    result = {
        "metric": "decoder-shaped shard GEMMs (hidden 4096, FFN 11008 / 8)", "value": big["gate_up_tflops"],
        "unit": "TFLOP/s", "n_gpus": 1, "higher_is_better": True, "dtype": "bf16", "data": "synthetic",
        "config": {"workload": "gate/up [M,4096]x[4096,1376] all-scatter to 8 ranks + down [M,1376]x[1376,4096] "
                               "fp32 partial + one-shot reduce of 8 partials; value = gate/up at M=2048"},
        "per_M": rows,
    }
    if emit:
        print(json.dumps(result))
    return result


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py measures one GPU's share of the path; --gpus {args.gpus} is not supported "
              "(no collectives or multi-GPU runs are part of this build).", file=sys.stderr)
        sys.exit(2)

    import torch

    import iris_amd
    from iris_amd import ops

    if not torch.cuda.is_available():
        print("bench.py needs a GPU", file=sys.stderr)
        sys.exit(1)
    if args.workload == "atomic":
        return run_atomic(args)
    if args.workload == "decoder":
        return run_decoder(args)
    if args.workload == "shapes":
        return run_shapes(args)
    if args.workload == "fp32":
        return run_fp32(args)
    if args.workload == "fused":
        return run_fused(args)

    ws = 8
    # per-rank heap: full-K operands 2 x 128 MiB, bf16 results 2 x 128 MiB, fp32 partial 256 MiB, flags
    shmem = iris_amd.iris(1 << 30, virtual_ranks=ws)
    dtype = torch.bfloat16
    g = torch.Generator().manual_seed(123)
    # one rank's K-shard as a strided view of the full-K operands (the 08/09 sharding)
    A_full = (torch.randn(M, K_TOTAL, generator=g) * 0.02).to(dtype)
    B_full = (torch.randn(N, K_TOTAL, generator=g) * 0.02).to(dtype)
    if args.zero_operands:
        A_full.zero_()
        B_full.zero_()
    if args.offheap_operands:
        a_full, bt_full = A_full.cuda(), B_full.cuda()
    else:
        a_full = shmem.zeros((M, K_TOTAL), dtype=dtype)
        a_full.copy_(A_full)
        bt_full = shmem.zeros((N, K_TOTAL), dtype=dtype)
        bt_full.copy_(B_full)
    a = a_full[:, :K_SHARD]
    b = bt_full[:, :K_SHARD].T
    del A_full, B_full
    c_global = shmem.zeros((M, N), dtype=dtype)
    total_tiles = ops.cdiv(M, BLK_M) * ops.cdiv(N, BLK_N)
    flags = shmem.zeros((total_tiles,), dtype=torch.int32)
    hb = shmem.get_heap_bases()
    num_xcds = ops.default_num_xcds(shmem.get_cu_count(), GRID)

    def gemm_on(x, y):
        ops.gemm_launch(x, y, None, c_global, flags, hb, 0, 1, GRID, BLK_M, BLK_N, BLK_K, args.gsize_m,
                        ops.EPI_ALL_SCATTER, notify=True, num_xcds=num_xcds, variant=args.variant)

    def gemm_step():
        gemm_on(a, b)

    flops = 2.0 * M * N * K_SHARD
    settle_launches = 0
    t_end = time.perf_counter() + args.settle_ms * 1e-3
    while time.perf_counter() < t_end:
        for _ in range(20):
            gemm_step()
        torch.cuda.synchronize()
        settle_launches += 20
    wall, kernel_ms = timed_steps(gemm_step, args.steps, args.warmup)
    ms_per_step = wall / args.steps * 1e3
    tflops = flops / (ms_per_step * 1e-3) / 1e12
    kernel_tflops = flops / (kernel_ms * 1e-3) / 1e12
    assert int(flags.min().item()) == int(flags.max().item()) == args.steps + args.warmup + settle_launches, \
        "every tile publishes once per step"
    regs, spills = ops.gemm_kernel_info(a, b, None, c_global, flags, hb, 0, 1, GRID, BLK_M, BLK_N, BLK_K,
                                        args.gsize_m, ops.EPI_ALL_SCATTER, num_xcds=num_xcds, variant=args.variant)

    details = {}  # printed before the result line, one JSON line per entry
    result = {
        "metric": "fused GEMM+reduce TFLOP/s (% bf16 MFMA peak); reduce-phase HBM GB/s",
        "value": round(tflops, 2),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "settle_ms": args.settle_ms,
        "ms_per_step": round(ms_per_step, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic, all-zero operands (a measurement of the kernel's structure, not the metric's workload)"
                if args.zero_operands else "synthetic",
        "config": {
            "workload": "single-shard fused GEMM + flag-published epilogue: bf16 A[8192,1024] x B[1024,8192] "
                        "(K-shard views, lda=ldb=8192), fp32 accumulate, 256x256 tiles -> bf16 in the fine-grained "
                        "heap, one uint32 ready flag per tile",
            "M": M, "N": N, "K_shard": K_SHARD, "BLK_M": BLK_M, "BLK_N": BLK_N, "gsize_m": args.gsize_m,
            "grid": GRID, "num_xcds": num_xcds, "variant": args.variant,
            "operands": "device memory outside the heap" if args.offheap_operands else "fine-grained heap",
        },
        "pct_of_bf16_peak": round(100.0 * tflops / PEAK_BF16_TFLOPS, 2),
        "gemm_kernel": {"registers": regs, "spill_bytes": spills, "mean_ms": round(kernel_ms, 5)},
        "roofline": {
            "bound": "mfma",
            "achieved": round(kernel_tflops, 2),
            "peak": PEAK_BF16_TFLOPS,
            "unit": "TFLOP/s",
            "frac": round(kernel_tflops / PEAK_BF16_TFLOPS, 4),
            "traffic": GEMM_TRAFFIC_BYTES if args.variant == 0 and args.gsize_m == GSIZE_M else None,
        },
    }

    if not args.no_coldcache:
        # the reference's own timing protocol (iris/util.py:62-104): every repetition starts behind a 256 MiB
        # cache flush and a device synchronise, one event pair per launch
        cold_ms = iris_amd.do_bench(gemm_step, shmem.barrier, lambda: None, n_warmup=10, n_repeat=50)
        cold_tflops = flops / (cold_ms * 1e-3) / 1e12
        result["gemm_cold_cache"] = {"protocol": "do_bench: 256 MiB cache flush before every repetition, mean of 50",
                                     "ms": round(cold_ms, 5), "tflops": round(cold_tflops, 2),
                                     "frac": round(cold_tflops / PEAK_BF16_TFLOPS, 4)}
        if not args.no_context:
            # the vendor library's GEMM on the same operands under the same protocol (no flags)
            lib_out = torch.empty((M, N), dtype=dtype, device="cuda")
            lib_cold_ms = iris_amd.do_bench(lambda: torch.matmul(a, b, out=lib_out), shmem.barrier, lambda: None,
                                            n_warmup=10, n_repeat=50)
            result["gemm_cold_cache"]["library_ms"] = round(lib_cold_ms, 5)
            result["gemm_cold_cache"]["library_tflops"] = round(flops / (lib_cold_ms * 1e-3) / 1e12, 2)
            del lib_out

    if not args.no_reduce:
        # reduce phase: 8 fp32 partials [8192,8192] (one per virtual rank) -> bf16
        c = shmem.zeros((M, N), dtype=torch.float32)
        out = shmem.zeros((M, N), dtype=dtype)
        for r in range(ws):
            part = shmem.on_rank(c, r)
            part.normal_(generator=None)
            shmem.on_rank(flags, r).zero_()
        torch.cuda.synchronize()

        # One set of tile flags per timed launch, all armed beforehand (the
        # producers' signals: +1 on every other rank's flags), so that the
        # timed region holds nothing but the reduce launches, back to back
        # under one event pair like the GEMM's.
        steps = max(5, min(args.steps, 30))
        flag_sets = [shmem.zeros((total_tiles,), dtype=torch.int32) for _ in range(3 + steps)]
        for f in flag_sets:
            for r in range(ws):
                shmem.on_rank(f, r).zero_()
        for f in flag_sets:
            for r in range(ws):
                ops.signal_tiles(shmem.on_rank(f, r), hb, total_tiles, r, ws)
        torch.cuda.synchronize()
        for f in flag_sets[:3]:
            ops.one_shot_reduce(c, out, f, hb, 0, ws, BLK_M, BLK_N, args.gsize_m, variant=args.reduce_variant)
        torch.cuda.synchronize()
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record()
        for f in flag_sets[3:]:
            ops.one_shot_reduce(c, out, f, hb, 0, ws, BLK_M, BLK_N, args.gsize_m, variant=args.reduce_variant)
        e.record()
        torch.cuda.synchronize()
        red_ms = [s.elapsed_time(e) / steps]
        for f in flag_sets:
            assert int(f.abs().max().item()) == 0, "the reduce consumes every flag"
        assert int(flags.abs().max().item()) == 0, "the reduce consumes every flag"
        rbytes = ws * M * N * 4 + M * N * 2
        rms = statistics.mean(red_ms)
        gbps = rbytes / (rms * 1e-3) / 1e9
        # the reduce half of the metric, inside `roofline` so that it travels with the GEMM's
        result["roofline"]["reduce"] = {
            "workload": "one-shot reduce of 8 fp32 partial-C [8192,8192] -> bf16, gated by per-tile flags",
            "bound": "hbm", "achieved": round(gbps, 1), "peak": PEAK_HBM_GBPS, "unit": "GB/s",
            "frac": round(gbps / PEAK_HBM_GBPS, 4),
            "traffic": REDUCE_TRAFFIC_BYTES if args.reduce_variant == 0 else None,
            "ms": round(rms, 5), "launches": steps, "variant": args.reduce_variant,
        }
        result["reduce_GBps"] = round(gbps, 1)
        result["pct_of_hbm_peak"] = round(100.0 * gbps / PEAK_HBM_GBPS, 2)
        if not args.no_context:
            # the same launch with other numbers of groups (the default is two per CU): the rate follows the
            # groups a CU hosts, not the bytes it requests; 10 launches each, flags armed beforehand as above
            sweep = {}
            cus = shmem.get_cu_count()
            for groups in (cus, cus * 3 // 2, cus * 2, cus * 3):
                fs = flag_sets[:13]
                for f in fs:
                    for r in range(ws):
                        ops.signal_tiles(shmem.on_rank(f, r), hb, total_tiles, r, ws)
                for f in fs[:3]:
                    ops.one_shot_reduce(c, out, f, hb, 0, ws, BLK_M, BLK_N, args.gsize_m, num_sms=groups)
                torch.cuda.synchronize()
                s.record()
                for f in fs[3:]:
                    ops.one_shot_reduce(c, out, f, hb, 0, ws, BLK_M, BLK_N, args.gsize_m, num_sms=groups)
                e.record()
                torch.cuda.synchronize()
                sweep[str(groups)] = round(rbytes / (s.elapsed_time(e) / 10 * 1e-3) / 1e9 / PEAK_HBM_GBPS, 4)
            details["reduce_frac_by_groups"] = sweep

    if not args.no_context:
        # (after the two headline measurements: seconds of probes at the power cap in front of the reduce's
        # thirty launches would be measured with them)
        ctx = context_figures(a, b, c_global, flops, gemm_on)
        details["context"] = ctx
        # the one-line version for the result line: the vendor library's plain GEMM on the same operands, this
        # kernel and the library on zeros, what the matrix cores alone sustain on such data
        result["context"] = {
            "library_gemm_ms": ctx["library_gemm"]["ms"],
            "gemm_on_zeros_ms": ctx["gemm_on_zeros"]["ms"],
            "library_gemm_on_zeros_ms": ctx["library_gemm_on_zeros"]["ms"],
            "mfma_only_tflops_on_such_data": ctx["mfma_sustained[random N(0,0.02)]"]["tflops"],
            "mfma_only_tflops_on_zeros": ctx["mfma_sustained[zeros]"]["tflops"],
            "shader_clock_mhz": {k: v for k, v in ctx["shader_clock_mhz"].items() if k != "how"},
        }

    if args.copy_calibration:
        # ws=1, fp32 -> fp32: the reduce kernel degenerates to a plain tiled copy
        src = torch.randn((M, N), dtype=torch.float32, device="cuda")
        dst = torch.zeros((M, N), dtype=torch.float32, device="cuda")
        for _ in range(3):
            ops.one_shot_reduce(src, dst, flags, hb, 0, 1, BLK_M, BLK_N, args.gsize_m, wait_flags=False)
        torch.cuda.synchronize()
        assert torch.equal(src, dst)
        result["copy_calibration"] = {"kernel": "reduce_tiles_vec_kernel<fp32, fp32, ws=1>",
                                      "read_bytes": M * N * 4, "write_bytes": M * N * 4, "launches": 3}

    if not args.no_context and not args.no_other_workloads:
        # the other configurations, each measured as its own --workload run measures it
        at = run_atomic(args, emit=False)
        dec = run_decoder(args, emit=False)
        keep = ("M", "kernel_up", "split_k_up", "gate_up_us", "gate_up_tflops", "gate_up_weight_GBps", "kernel_down",
                "split_k_down", "down_us", "down_tflops", "reduce_us", "reduce_GBps", "gate_up_one_destination_us",
                "gate_up_without_fetching_waves_us",
                "library_gate_up_us", "library_down_us", "at_reference_default_tile_256x64")
        args.shapes_gpus = "8"  # (the whole sweep, 1 to 8 GPUs, is the --workload shapes run)
        sweep = run_shapes(args, emit=False)
        fz = run_fused(args, emit=False)
        f32 = run_fp32(args, emit=False)
        details["other_workloads"] = {
            "atomic_accumulate": {k: at[k] for k in ("value", "unit", "ms_per_step", "atomic_updates_per_s",
                                                     "atomic_ceiling", "config")},
            "decoder_shards": {"config": dec["config"], "per_M": [{k: r[k] for k in keep} for r in dec["per_M"]]},
            "shape_sweep_8_gpus": {"vs_library_geomean": sweep["value"], "worst": sweep["worst"],
                                   "best": sweep["best"], "config": sweep["config"],
                                   "points": [{k: pt[k] for k in ("algorithm", "shard", "tile", "kernel", "split_k",
                                                                  "us", "tflops", "library_us", "vs_library")}
                                              for pt in sweep["points"]]},
            "one_shot_in_program": {k: fz[k] for k in ("config", "in_program", "two_kernels",
                                                       "in_program_vs_two_kernels", "checked")},
            "fp32_operands": {k: f32[k] for k in ("config", "kernel", "value", "unit", "ms_per_step", "roofline",
                                                  "library_ms", "library_tflops")},
        }
        # one line each for the result line
        result["other_workloads"] = {
            "atomic_accumulate_ms": at["ms_per_step"],
            "atomic_frac_of_atomic_ceiling": at["atomic_ceiling"]["frac_of_ceiling"],
            "decoder_gate_up_us_by_M": {str(r["M"]): r["gate_up_us"] for r in dec["per_M"]},
            "decoder_library_gate_up_us_by_M": {str(r["M"]): r["library_gate_up_us"] for r in dec["per_M"]},
            "decoder_down_us_by_M": {str(r["M"]): r["down_us"] for r in dec["per_M"]},
            "decoder_library_down_us_by_M": {str(r["M"]): r["library_down_us"] for r in dec["per_M"]},
            "shape_sweep_8_gpus_vs_library": {"geomean": sweep["value"], "worst": sweep["worst"],
                                              "best": sweep["best"]},
            "one_shot_in_program_2_ranks_ms": fz["in_program"]["ms"],
            "one_shot_two_kernels_2_ranks_ms": fz["two_kernels"]["ms"],
            "fp32_operands_tflops": f32["value"],
            "fp32_operands_library_tflops": f32["library_tflops"],
        }

    if not args.no_cpu:
        result["cpu_baseline"] = cpu_baseline()

    # the groups of detail first, one line each; the result line last
    for name, value in details.items():
        print(json.dumps({"detail": name, name: value}))
    sys.stdout.flush()
    print(json.dumps(result))


if __name__ == "__main__":
    main()
