"""The tiles, cells and few-rows builds for a row-major B (``_rows``) and for operands along K at any alignment (``_gather_dma``)
where other ranks wait for them: a one-shot product's partials, flags and reduce, inside the program and behind it, stores to
several ranks, blocks that share K, split last rounds, columns apart and parts of tiles, against the CPU oracle."""

import pytest
import torch

from iris_amd import ops
from oracle import iris_oracle as O
from parity import check_close, make_ab
from test_gemm_gather_gpu import place

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def operands(shmem, M, N, K, dtype):
    """A row-major B."""
    A, B = make_ab(M, N, K, dtype)
    return A, B, place(shmem, A, False, 0, 0), place(shmem, B, False, 0, 0)


def loose_operands(shmem, M, N, K, dtype):
    """An odd K: rows off the 16 bytes."""
    A, B = make_ab(M, N, K, dtype)
    return A, B, place(shmem, A, False, 0, 0), place(shmem, B.T, False, 0, 0).T


GATHER = "128x128x64_w2x2_gather+reduce", "64x64x128_w2x2_gather+reduce"


@pytest.mark.parametrize("rows,M,N,ks,BM,BN,part,ws,grid,name,fused", [
    # fewer programs than CUs: whole tiles, the reduce inside
    (True, 300, 264, 200, 256, 128, F32, 4, 64, "256x128x64_w2x2_s3_f4_rows", GATHER[0]),
    (True, 520, 512, 136, 256, 256, BF16, 3, 64, "256x256x64_w2x4_s2_rows", GATHER[0]),
    (False, 300, 264, 201, 256, 128, F32, 4, 64, "256x128x64_w2x2_s3_f4_gather_dma", GATHER[0]),
    (False, 513, 300, 131, 256, 256, BF16, 3, 64, "256x256x64_w2x4_s2_gather_dma", GATHER[0]),
    # cells and few rows, on both sides of where the reduce goes behind them
    (True, 300, 264, 520, 128, 128, F32, 2, 256, "cells_32x32_rows", None),
    (True, 300, 264, 136, 64, 64, BF16, 4, 256, "cells_32x32_rows", GATHER[1]),
    (True, 13, 1376, 520, 64, 64, BF16, 4, 256, "cells_16x32_rows", None),
    (False, 300, 264, 1543, 64, 64, BF16, 4, 256, "cells_32x32_gather_dma", None),
    (False, 300, 264, 133, 64, 64, BF16, 4, 256, "cells_32x32_gather_dma", GATHER[1]),
    (False, 9, 700, 1031, 64, 64, F32, 4, 256, "few_rows_16xN_gather_dma", None),
    (False, 16, 512, 133, 64, 64, F32, 2, 256, "few_rows_16xN_gather_dma", GATHER[1]),
])
@pytest.mark.parametrize("last", [ops.PHASE_FUSED, ops.PHASE_TWO_KERNELS])
def test_one_shot(shmem, rows, M, N, ks, BM, BN, part, ws, grid, name, fused, last):
    """Every rank but the last produces; the last produces, waits for the others' flags and reduces."""
    A, B, a, b = (operands if rows else loose_operands)(shmem, M, N, ks * ws, BF16)
    shards = O.k_shards(A, B, ws)
    c, cg = shmem.zeros((M, N), dtype=part), shmem.zeros((M, N), dtype=BF16)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total,), dtype=torch.int32)
    P, locks = shmem.zeros((grid, BM * BN), dtype=F32), shmem.zeros((grid,), dtype=torch.int32)
    for r in range(ws):
        for t in (c, cg, flags):
            shmem.on_rank(t, r).zero_()
    for r in range(ws):
        args = (a[:, r * ks:(r + 1) * ks], b[r * ks:(r + 1) * ks, :], shmem.on_rank(c, r), shmem.on_rank(cg, r),
                shmem.on_rank(flags, r), shmem.get_heap_bases(), r, ws, grid, BM, BN, 64, 6, ops.EPI_ONE_SHOT)
        kw = dict(phase=last if r == ws - 1 else ops.PHASE_PRODUCE, partials=P, locks=locks, num_xcds=8)
        inside = kw["phase"] == ops.PHASE_FUSED
        assert ops.gemm_plan_name(*args, **kw) == ((fused or name + "+kernel+reduce") if inside else name)
        ops.gemm_launch(*args, **kw)
    torch.cuda.synchronize()
    for r in range(ws):
        check_close(shmem.on_rank(c, r), O.shard_gemm(*shards[r], part), f"partial {r}")
        assert shmem.on_rank(flags, r).cpu().tolist() == [0 if r == ws - 1 else ws - 1] * total
    got = torch.stack([shmem.on_rank(c, r).cpu() for r in range(ws)])
    assert torch.equal(shmem.on_rank(cg, ws - 1).cpu(), O.one_shot_reduce(got, BF16))
    assert not locks.any()


ROWS, LOOSE = "_rows", "_gather_dma"


@pytest.mark.parametrize("rows,M,N,K,BM,BN,ws,grid,name,parts", [
    # tiles to several ranks
    (True, 600, 520, 264, 256, 128, 4, 64, "256x128x64_w2x2_s3_f4%s", 1),
    (False, 600, 523, 265, 256, 256, 4, 64, "256x256x64_w2x4_s2%s", 1),
    # blocks of the caller's tiles, K in two
    (True, 1024, 256, 4096, 256, 64, 1, 16, "256x128x64_w2x2_s3_f4%s+two_tiles_each", 2),
    (False, 1024, 256, 4097, 256, 64, 2, 16, "256x128x64_w2x2_s3_f4%s+two_tiles_each", 2),
    (True, 1024, 512, 4096, 256, 128, 2, 16, "256x256x64_w2x4_s2%s+two_tiles_each", 2),
    (False, 1000, 512, 4097, 256, 128, 1, 16, "256x256x64_w2x4_s2%s+two_tiles_each", 2),
    # a last round that is shared out
    (True, 1024, 384, 4096, 128, 128, 2, 16, "128x128x64_w2x2_s4_f4%s+last_round_in_2_parts", 1),
    (False, 1000, 384, 4099, 128, 128, 1, 16, "128x128x64_w2x2_s4_f4%s+last_round_in_2_parts", 1),
    # a column of tiles apart
    (True, 1024, 320, 4096, 256, 64, 2, 16, "256x128x64_w2x2_s3_f4%s+two_tiles_each+last_64_columns_apart", 2),
    (False, 1024, 320, 4097, 256, 64, 1, 16, "256x128x64_w2x2_s3_f4%s+two_tiles_each+last_64_columns_apart", 2),
    # parts of tiles, alone and with K shared
    (True, 300, 200, 192, 256, 256, 2, 256, "64x64x128_w2x2_s4_f4%s+parts_of_tiles", 1),
    (True, 200, 144, 2048, 128, 128, 3, 256, "64x64x128_w2x2_s4_f4%s+parts_of_tiles", 8),
    (False, 300, 200, 193, 256, 256, 2, 256, "64x64x128_w2x2_s4_f4%s+parts_of_tiles", 1),
    (False, 200, 140, 2049, 128, 128, 3, 256, "64x64x128_w2x2_s4_f4%s+parts_of_tiles", 8),
])
def test_scatter(shmem, rows, M, N, K, BM, BN, ws, grid, name, parts):
    A, B, a, b = (operands if rows else loose_operands)(shmem, M, N, K, F16)
    cg = shmem.zeros((M, N * ws), dtype=F16)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total + 1,), dtype=torch.int32)
    P, locks = shmem.zeros((grid, BM * BN), dtype=F32), shmem.zeros((grid,), dtype=torch.int32)
    for r in range(ws):
        shmem.on_rank(cg, r).zero_()
        shmem.on_rank(flags, r).zero_()
    args = (a, b, None, cg, flags, shmem.get_heap_bases(), 0, ws, grid, BM, BN, 64, 4, ops.EPI_ALL_SCATTER)
    # (one XCD: small products in parts, not cells)
    kw = dict(partials=P, locks=locks, num_xcds=1 if "parts_of" in name else 8)
    assert ops.gemm_plan_name(*args, **kw) == name % (ROWS if rows else LOOSE) and ops.gemm_split_k(*args, **kw) == parts
    want = O.shard_gemm(A, B, F16)
    for launch in (1, 2):
        ops.gemm_launch(*args, **kw)
        torch.cuda.synchronize()
        for r in range(ws):
            check_close(shmem.on_rank(cg, r)[:, :N], want, f"launch {launch}, rank {r}")
            assert shmem.on_rank(flags, r).cpu().tolist() == [launch] * total + [0]
        assert not locks.any()
