"""The work that users of this package have it do, as cases to be timed.

One rank of a tensor-parallel layer multiplies its shard and publishes the
result to its peers, in one of the package's three ways:

* ``all_scatter``  the shard's columns go to every rank, one ready flag a tile;
* ``atomics``      the K-shards are added up in C with atomics;
* ``one_shot``     partial sums are left in the heap, signalled tile by tile,
                   and every rank adds all ranks' partials up.

The ranks are sub-heaps of the one GPU (``iris.iris(..., virtual_ranks=P)``);
activations and weights are the program's own tensors, everything that peers
touch lives in the symmetric heap.  A pass is what a program does for one
layer: re-arm the flags, launch, reduce.
"""

import math

import torch

import iris_amd as iris
from iris_amd import ops
from iris_amd.matmul import matmul_all_scatter, matmul_atomics_all_reduce, matmul_one_shot_all_reduce

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SIZES = {"bf16": 2, "fp16": 2, "fp32": 4}
PROGRAMS = 256  # the examples' --gemm_sms: one persistent program per CU


def _case(name, path, m, n, k, ranks, dtype, tile, gsize, partial="", out="", weight="nk", phase=""):
    """``n`` and ``k`` are the rank's shard.  ``weight``: "nk" for weights kept as [n, k] rows and passed
    transposed (a linear layer's forward), "kn" for row-major [k, n] (the same weights in the backward product for
    the activations, or a layer that stores them so)."""
    case = {"path": path, "m": m, "n": n, "k": k, "ranks": ranks, "dtype": dtype, "tile_m": tile[0], "tile_n": tile[1],
            "gsize": gsize, "partial": partial or dtype, "out": out or dtype, "weight": weight, "phase": phase}
    return dict(case, name=name) if name else case


def listed():
    return [
        # One token through the gate / up projection of a 6.7B decoder cut over eight ranks: the smallest call there
        # is in serving, all latency and host time.
        _case("decode_1", "all_scatter", 1, 1376, 4096, 8, "bf16", (64, 64), 4),
        # A batch of sixteen tokens through the same decoder's down projection: a K-shard, its partial sums and
        # the reduce behind it.
        _case("decode_16_down", "one_shot", 16, 4096, 1376, 8, "bf16", (64, 64), 6, partial="fp32", phase="two_kernels"),
        # A short prompt, 128 tokens, gate / up.
        _case("prompt_128", "all_scatter", 128, 1376, 4096, 8, "bf16", (64, 64), 4),
        # A prompt of a length that fits no tile, down projection, the one-shot entry point as it is called by default
        # (the reduce inside the program), 16-bit partials as the example script allocates them.
        _case("prompt_1999_down", "one_shot", 1999, 4096, 1376, 8, "bf16", (256, 128), 6, phase="fused"),
        # Rows, columns and depth that are multiples of nothing, at the example script's tile.
        _case("odd_sizes", "all_scatter", 1000, 999, 1500, 2, "fp16", (256, 64), 4),
        # Weights in row-major order: what the backward pass for the activations of a linear layer multiplies with.
        _case("row_major_weight", "all_scatter", 2048, 1376, 4096, 1, "bf16", (256, 128), 4, weight="kn"),
        # fp32 operands (the scripts' --datatype fp32) at the default tile.
        _case("fp32", "all_scatter", 2048, 2048, 1024, 1, "fp32", (256, 64), 4),
        # A K-shard of a training-sized product, 256 x 256 tiles with a ready flag each: the benchmark's headline.
        _case("shard_8192", "all_scatter", 8192, 8192, 1024, 1, "bf16", (256, 256), 4),
        # Eight K-shards added into one fp32 C.
        _case("atomics_4096", "atomics", 4096, 4096, 512, 8, "bf16", (256, 256), 6, out="fp32"),
        # The example script of the all-scatter as it comes: fp16, 256 x 64 tiles, its default problem over 8 ranks.
        _case("script_default", "all_scatter", 8192, 576, 36864, 8, "fp16", (256, 64), 4),
        # The one-shot all-reduce as the example script runs it on one GPU: every rank produces, every rank reduces.
        _case("allreduce_4_ranks", "one_shot_ranks", 8192, 4096, 3584, 4, "bf16", (256, 128), 6),
        # The reduce alone: eight fp32 partials that producers left in the heap, flags raised.
        _case("reduce_8192", "reduce", 8192, 8192, 0, 8, "bf16", (256, 256), 4, partial="fp32"),
    ]


# the largest listed case's operations, and what matrix cores do at a sixteenth of the 16-bit rate
_MOST_FLOPS, _MOST_FLOPS_FP32 = 9.0e11, 3.4e10
_MOST_ELEMENTS = 1 << 26  # of one rank's output


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extent(rng, lo, hi, odd):
    """A length between lo and hi: mostly a multiple of 64 or of 8, an arbitrary one in ``odd`` of the cases."""
    v, r = _log(rng, lo, hi), rng.random()
    step = 1 if r < odd else 8 if r < 0.5 else 64
    return max(lo, v // step * step)


def draw(rng):
    while True:
        path = rng.choices(["all_scatter", "one_shot", "one_shot_ranks", "atomics", "reduce"], [45, 22, 10, 13, 10])[0]
        dtype = rng.choices(["bf16", "fp16", "fp32"], [55, 30, 15])[0]
        ranks = rng.choice([1, 2, 4, 8] if path == "all_scatter" else [2, 4, 8])
        m = _log(rng, 1, 8192)
        n = _extent(rng, 128, 8192, 0.15)
        k = 0 if path == "reduce" else _extent(rng, 128, 36864, 0.1)
        # small tiles for a few rows, the scripts' and the sweep's tiles for many
        tile = rng.choice([(64, 64), (128, 128), (256, 64)] if m <= 512 else [(256, 64), (256, 128), (256, 256), (128, 128)])
        gsize = 4 if path in ("all_scatter", "reduce") else 6
        partial = dtype if dtype == "fp32" or rng.random() < 0.5 else "fp32"
        out = partial if path == "atomics" else dtype
        phase = rng.choice(["fused", "two_kernels"]) if path == "one_shot" else ""
        weight = "kn" if path != "reduce" and rng.random() < 0.12 else "nk"
        shards = ranks if path in ("one_shot_ranks", "atomics") else 1
        flops = 2.0 * m * n * k * shards
        if flops > (_MOST_FLOPS_FP32 if dtype == "fp32" else _MOST_FLOPS):
            continue
        if m * n * (ranks if path == "all_scatter" else 1) > _MOST_ELEMENTS:
            continue
        return _case(None, path, m, n, k, ranks, dtype, tile, gsize, partial, out, weight, phase)


def _operands(case, gen, shards):
    """(activations [m, k], weights [k, n]) of ``shards`` consecutive K-shards, as views of the whole operands."""
    dtype, k = DTYPES[case["dtype"]], case["k"]
    x = torch.empty((case["m"], k * shards), device="cuda", dtype=dtype).normal_(0.0, 0.05, generator=gen)
    if case["weight"] == "nk":
        w = torch.empty((case["n"], k * shards), device="cuda", dtype=dtype).normal_(0.0, 0.05, generator=gen).T
    else:
        w = torch.empty((k * shards, case["n"]), device="cuda", dtype=dtype).normal_(0.0, 0.05, generator=gen)
    return [(x[:, r * k:(r + 1) * k], w[r * k:(r + 1) * k, :]) for r in range(shards)]


def prepare(case, seed):
    m, n, ranks, path = case["m"], case["n"], case["ranks"], case["path"]
    tm, tn = case["tile_m"], case["tile_n"]
    tiles = ops.cdiv(m, tm) * ops.cdiv(n, tn)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    wide = n * ranks if path == "all_scatter" else n
    heap = (m * wide * SIZES[case["out"]] + m * n * SIZES[case["partial"]] + 4 * tiles + 4 * PROGRAMS * (tm * tn + 1) + (1 << 20))
    heap = (heap + 0xFFFFF) & ~0xFFFFF
    world = 1 if path == "atomics" else ranks  # (the K-shards of "atomics" meet in one C)
    shmem = iris.iris(heap, virtual_ranks=world)
    rank = world // 2  # the rank whose share is run where one rank's is
    state = {"case": case, "shmem": shmem, "rank": rank, "world": world, "bases": shmem.get_heap_bases(),
             "cus": shmem.get_cu_count()}
    result = shmem.zeros((m, wide), dtype=DTYPES[case["out"]])
    flags = shmem.zeros((tiles,), dtype=torch.int32)
    state["result"] = [shmem.on_rank(result, r) for r in range(world)]
    state["flags"] = [shmem.on_rank(flags, r) for r in range(world)]
    for r in range(world):
        state["result"][r].zero_()
        state["flags"][r].zero_()
    if path == "reduce":
        state["shards"] = []
    else:
        state["shards"] = _operands(case, gen, ranks if path in ("one_shot_ranks", "atomics") else 1)
        # the workspace that the example scripts allocate beside the operands
        state["P"] = shmem.zeros((PROGRAMS, tm * tn), dtype=torch.float32)
        state["locks"] = shmem.zeros((PROGRAMS,), dtype=torch.int32)
        for matmul in (matmul_all_scatter, matmul_atomics_all_reduce, matmul_one_shot_all_reduce):
            matmul.set_debug(False)
    if path in ("one_shot", "one_shot_ranks", "reduce"):
        partial = shmem.zeros((m, n), dtype=DTYPES[case["partial"]])
        state["partial"] = [shmem.on_rank(partial, r) for r in range(world)]
        for r in range(world):
            if path == "one_shot_ranks":
                state["partial"][r].zero_()
            else:  # what the peers have computed
                state["partial"][r].normal_(0.0, 0.05 * math.sqrt(max(case["k"], 400) / 400.0), generator=gen)
    else:
        state["partial"] = [None] * world
    return state


def _apply(matmul, state, shard, rank):
    case = state["case"]
    a, b = state["shards"][shard]
    matmul.apply(a, b, state["partial"][rank], state["result"][rank], None, state["P"], state["locks"],
                 state["flags"][rank], rank, state["world"], PROGRAMS, case["tile_m"], case["tile_n"], 64, case["gsize"],
                 "True", 2, 8, 0, 16, 2, state["bases"], state["cus"])


def run(state):
    case, rank, world = state["case"], state["rank"], state["world"]
    path = case["path"]
    if path == "all_scatter":
        iris.memset_tensor(state["flags"][rank], 0)
        _apply(matmul_all_scatter, state, 0, rank)
        return {"result": state["result"], "flags": state["flags"][rank]}
    if path == "atomics":
        state["result"][0].zero_()
        for shard in range(case["ranks"]):
            _apply(matmul_atomics_all_reduce, state, shard, 0)
        return {"result": state["result"][0]}
    if path == "one_shot":
        # the peers have produced and signalled; this rank produces, signals and reduces
        iris.memset_tensor(state["flags"][rank], world - 1)
        matmul_one_shot_all_reduce.phase = ops.PHASE_FUSED if case["phase"] == "fused" else ops.PHASE_TWO_KERNELS
        _apply(matmul_one_shot_all_reduce, state, 0, rank)
        return {"result": state["result"][rank], "partial": state["partial"][rank], "flags": state["flags"][rank]}
    if path == "one_shot_ranks":
        for phase in (ops.PHASE_PRODUCE, ops.PHASE_CONSUME):
            matmul_one_shot_all_reduce.phase = phase
            for r in range(world):
                _apply(matmul_one_shot_all_reduce, state, r, r)
        return {"result": state["result"], "partial": state["partial"], "flags": state["flags"]}
    iris.memset_tensor(state["flags"][rank], world - 1)
    ops.one_shot_reduce(state["partial"][rank], state["result"][rank], state["flags"][rank], state["bases"], rank, world,
                        case["tile_m"], case["tile_n"], case["gsize"], num_xcds=8)
    return {"result": state["result"][rank], "flags": state["flags"][rank]}


def work(case):
    m, n, k, ranks, path = case["m"], case["n"], case["k"], case["ranks"], case["path"]
    shards = ranks if path in ("one_shot_ranks", "atomics") else 1
    operands = shards * (m * k + k * n) * SIZES[case["dtype"]]
    partial, out = m * n * SIZES[case["partial"]], m * n * SIZES[case["out"]]
    moved = {
        "all_scatter": ranks * out,          # the shard's columns on every rank
        "atomics": out,
        "one_shot": ranks * partial + out,   # the peers' partials in, this rank's out, and the sum
        "one_shot_ranks": ranks * (partial + out),
        "reduce": ranks * partial + out,
    }[path]
    return {"bytes": operands + moved, "flops": 2.0 * m * n * k * shards}


def tolerance(case):
    # The products are summed in fp32 in an order that is free, then rounded to the output's type: results may
    # differ by fp32 summation order, and by a last place where that carries a sum over a rounding boundary.
    if case["path"] == "reduce":
        kind = case["out"]
    else:
        kind = {"bf16", "fp16"} & {case["out"], case["partial"] if case["path"].startswith("one_shot") else case["out"]}
        kind = kind.pop() if kind else "fp32"
    return {"fp32": {"rel": 1e-5, "max": 2e-4}, "fp16": {"rel": 1e-3, "max": 4e-3}, "bf16": {"rel": 4e-3, "max": 2e-2}}[kind]
