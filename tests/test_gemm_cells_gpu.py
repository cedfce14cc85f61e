"""Small products in cells of 32 x 32 (one workgroup each, one round of them): values against the CPU oracle on every
rank, flags once per tile and launch, counters back at zero; edges in every direction, K shared out over workgroups,
each epilogue and operand type, and where the launcher keeps the tiles."""

import pytest
import torch

from iris_amd import ops
from oracle import iris_oracle as O
from parity import check_close, make_ab
from test_gemm_gather_gpu import place

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32
CELLS = "cells_32x32"


@pytest.mark.parametrize("M,N,K,BM,BN,ws,dtype,plan", [
    (65, 32, 8, 128, 32, 1, BF16, CELLS),        # a chunk of K; the last block of rows holds one
    (128, 1376, 4096, 64, 64, 2, BF16, CELLS),   # 4 x 43
    (100, 252, 1000, 128, 128, 1, F16, CELLS),   # ragged columns, a multiple of four
    (70, 45, 72, 256, 64, 3, BF16, CELLS),       # ... of nothing: rows of an odd length
    (213, 330, 648, 256, 256, 1, F16, CELLS),    # tiles larger than the matrix
    (1300, 190, 520, 256, 64, 1, BF16, CELLS),   # more rows than columns: dealt by rows
    (512, 512, 136, 64, 64, 1, BF16, CELLS),     # 256 cells
    (513, 512, 136, 64, 64, 1, BF16, None),      # 272: a second round
    (100, 96, 8200, 128, 64, 2, BF16, CELLS),    # 12 cells: K in parts
    (70, 64, 20000, 128, 64, 1, F16, CELLS),
    (150, 330, 1028, 64, 64, 1, F32, CELLS),
    (140, 60, 6004, 256, 64, 2, F32, CELLS),     # fp32, K in parts
    (100, 250, 333, 128, 128, 1, BF16, None),    # rows of A and B that start at any address
    (100, 250, 328, 80, 64, 1, BF16, None),      # a tile's rows are not whole cells
])
def test_scatter(shmem, M, N, K, BM, BN, ws, dtype, plan):
    A, B = make_ab(M, N, K, dtype)
    a, b = place(shmem, A, False, 0, 0), place(shmem, B.T, False, 0, 0).T
    cg = shmem.zeros((M, N * ws), dtype=dtype)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total + 2,), dtype=torch.int32)
    P, locks = shmem.zeros((256, 256 * 64), dtype=F32), shmem.zeros((256,), dtype=torch.int32)
    for r in range(ws):
        shmem.on_rank(cg, r).zero_()
        shmem.on_rank(flags, r).zero_()
    rank = ws - 1
    args = (a, b, None, shmem.on_rank(cg, rank), shmem.on_rank(flags, rank), shmem.get_heap_bases(), rank, ws, 256, BM, BN, 64,
            4, ops.EPI_ALL_SCATTER)
    kw = dict(partials=P, locks=locks, num_xcds=8)
    assert (ops.gemm_plan_name(*args, **kw) == CELLS) == (plan == CELLS)
    want = O.shard_gemm(A, B, dtype)
    for launch in (1, 2, 3):
        ops.gemm_launch(*args, **kw)
        torch.cuda.synchronize()
        for r in range(ws):
            check_close(shmem.on_rank(cg, r)[:, rank * N:], want, f"launch {launch}, rank {r}")
            assert shmem.on_rank(flags, r).cpu().tolist() == [launch] * total + [0, 0]
        assert not locks.any()
    assert not shmem.on_rank(cg, 0)[:, :rank * N].any()
    # without the counters' words the tiles stay, and so they do for a launch that shares the device
    assert ops.gemm_plan_name(*args, num_xcds=8) != CELLS or total > 256
    assert ops.gemm_plan_name(*args[:8], 248, *args[9:], num_xcds=8, partials=P, locks=locks) != CELLS


@pytest.mark.parametrize("dtype,part", [(BF16, F32), (F16, F16), (F32, F32)])
def test_one_shot_and_atomics(shmem, dtype, part):
    ws, M, N, ks, BM, BN = 4, 130, 200, 328, 128, 128
    A, B = make_ab(M, N, ks * ws, dtype)
    a, b = place(shmem, A, False, 0, 0), place(shmem, B.T, False, 0, 0).T
    shards = O.k_shards(A, B, ws)
    c, cg = shmem.zeros((M, N), dtype=part), shmem.zeros((M, N), dtype=dtype)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total,), dtype=torch.int32)
    acc = shmem.zeros((M, N), dtype=part)
    P, locks = shmem.zeros((256, BM * BN), dtype=F32), shmem.zeros((256,), dtype=torch.int32)
    for r in range(ws):
        for t in (c, cg, flags):
            shmem.on_rank(t, r).zero_()
    for r in range(ws):
        args = (a[:, r * ks:(r + 1) * ks], b[r * ks:(r + 1) * ks, :], shmem.on_rank(c, r), shmem.on_rank(cg, r),
                shmem.on_rank(flags, r), shmem.get_heap_bases(), r, ws, 256, BM, BN, 64, 6, ops.EPI_ONE_SHOT)
        kw = dict(phase=ops.PHASE_FUSED if r == ws - 1 else ops.PHASE_PRODUCE, partials=P, locks=locks, num_xcds=8)
        assert ops.gemm_plan_name(*args, **kw) == CELLS + ("+kernel+reduce" if r == ws - 1 else "")
        ops.gemm_launch(*args, **kw)
        ops.gemm_launch(args[0], args[1], None, acc, None, None, 0, 1, 256, BM, BN, 64, 6, ops.EPI_ATOMIC_ADD, num_xcds=8)
    torch.cuda.synchronize()
    for r in range(ws):
        check_close(shmem.on_rank(c, r), O.shard_gemm(*shards[r], part), f"partial {r}")
        assert shmem.on_rank(flags, r).cpu().tolist() == [0 if r == ws - 1 else ws - 1] * total
    check_close(shmem.on_rank(cg, ws - 1), O.one_shot_all_reduce(shards, part, dtype), "reduced")
    check_close(acc, O.shard_gemm(A, B, F32), "atomics")
    assert not locks.any()


@pytest.mark.parametrize("M,N,K,dtype,kind,name", [
    (92, 384, 32385, BF16, "loose", "cells_32x32_gather_dma"),     # 36 cells, five an XCD
    (40, 800, 18929, F16, "loose", "cells_32x32_gather_dma"),      # 50, seven an XCD
    (130, 160, 16384, BF16, "", "cells_32x32"),                    # 25
    (140, 224, 6004, F32, "", "cells_32x32"),                      # 35
    (27, 1120, 28032, BF16, "rows", "cells_32x32_rows"),           # 35 of a row-major B
    (5, 576, 36032, BF16, "rows", "cells_16x32_rows"),             # 18
])
def test_parts_of_k_fit_the_cus_of_each_xcd(shmem, M, N, K, dtype, kind, name):
    """A workgroup a CU: the parts of the cells that an XCD takes are all resident at once."""
    A, B = make_ab(M, N, K, dtype)
    a, b = place(shmem, A, False, 0, 0), place(shmem, B, False, 0, 0) if kind == "rows" else place(shmem, B.T, False, 0, 0).T
    cg = shmem.zeros((M, N), dtype=dtype)
    flags = shmem.zeros((ops.cdiv(M, 64) * ops.cdiv(N, 64),), dtype=torch.int32)
    P, locks = shmem.full((256, 256 * 64), float("nan"), dtype=F32), shmem.zeros((256,), dtype=torch.int32)
    args = (a, b, None, cg, flags, shmem.get_heap_bases(), 0, 1, 256, 64, 64, 64, 4, ops.EPI_ALL_SCATTER)
    kw = dict(partials=P, locks=locks, num_xcds=8)
    assert ops.gemm_plan_name(*args, **kw) == name
    ops.gemm_launch(*args, **kw)
    torch.cuda.synchronize()
    check_close(cg, O.shard_gemm(A, B, dtype), name)
    blocks = (1 if "16x32" in name else 2) * 2 * ops.cdiv(M, 32) * ops.cdiv(N, 32)  # of 16 x 16 sums, in register order
    parts, rest = divmod(int((~P.view(-1, 256).isnan()).any(dim=1).sum()), blocks)
    assert parts > 1 and rest == 0
    assert parts * ops.cdiv(ops.cdiv(M, 32) * ops.cdiv(N, 32), 8) <= torch.cuda.get_device_properties(0).multi_processor_count // 8
