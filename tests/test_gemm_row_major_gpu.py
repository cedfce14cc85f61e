"""The LDS-DMA tiles for a row-major B (``_rows``): every tile's edges, K steps that are whole, partial and single, padded
rows with NaN between them, split K, blocks of the caller's tiles, stores to one rank and atomics, against the CPU oracle; and the
forms that stay with the gathering tiles."""

import pytest
import torch

from iris_amd import ops
from oracle import iris_oracle as O
from parity import check_close, make_ab
from test_gemm_gather_gpu import place

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def operands(shmem, M, N, K, dtype, pad=0, shift=0):
    A, B = make_ab(M, N, K, dtype)
    return A, B, place(shmem, A, False, pad, shift), place(shmem, B, False, pad, shift)


@pytest.mark.parametrize("M,N,K,BM,BN,pad,shift,name", [
    (130, 72, 128, 64, 64, 0, 0, "64x64x128_w2x2_s4_f4_rows"),      # one K-step of 128
    (130, 200, 136, 64, 64, 8, 8, "64x64x128_w2x2_s4_f4_rows"),     # ... and one that holds a single chunk
    (64, 8, 8, 64, 64, 0, 0, "64x64x128_w2x2_s4_f4_rows"),          # the smallest
    (90, 64, 1544, 64, 64, 16, 0, "64x64x128_w2x2_s4_f4_rows"),
    (300, 136, 640, 128, 128, 0, 8, "128x128x64_w2x2_s4_f4_rows"),  # two tiles a program
    (257, 120, 72, 128, 64, 8, 0, "128x64x64_w2x2_s4_f4_rows"),
    (120, 264, 200, 64, 128, 0, 0, "64x128x64_w2x2_s4_f4_rows"),
    (520, 72, 456, 256, 64, 0, 0, "256x64x64_w4x1_s3_f4_rows"),
    (300, 200, 584, 256, 128, 0, 0, "256x128x64_w2x2_s3_f4_rows"),
    (513, 136, 1024, 256, 128, 24, 8, "256x128x64_w2x2_s3_f4_rows"),
    (513, 304, 200, 256, 256, 0, 0, "256x256x64_w2x4_s2_rows"),
    (300, 520, 1096, 256, 256, 8, 16, "256x256x64_w2x4_s2_rows"),
    (96, 200, 264, 64, 192, 0, 0, "64x64x128_w2x2_s4_f4_rows"),     # several compute tiles a logical tile
])
@pytest.mark.parametrize("dtype,out", [(BF16, BF16), (F16, F16), (BF16, F32)])
def test_scatter(shmem, M, N, K, BM, BN, pad, shift, name, dtype, out):
    A, B, a, b = operands(shmem, M, N, K, dtype, pad, shift)
    cg = shmem.full((M, N), 7, dtype=out)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total + 1,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, 3, BM, BN, 64, 2, ops.EPI_ALL_SCATTER)
    assert ops.gemm_plan_name(*args, variant=ops.VARIANT_PERSISTENT) == name
    for launch in (1, 2):
        ops.gemm_launch(*args, variant=ops.VARIANT_PERSISTENT)
        torch.cuda.synchronize()
        check_close(cg, O.shard_gemm(A, B, out), f"launch {launch}")
        assert flags.cpu().tolist() == [launch] * total + [0]


@pytest.mark.parametrize("M,N,K,BM,BN,parts", [
    (100, 200, 1032, 64, 64, 3),     # the owner's hand-over
    (100, 200, 1032, 64, 64, 8),     # sliced
    (256, 136, 1096, 128, 128, 4),
    (200, 72, 776, 256, 64, 4),
    (100, 264, 776, 64, 128, 3),
    (300, 248, 1032, 256, 128, 2),   # 128-accumulator tiles: the pair hand-over
    (300, 248, 1032, 256, 256, 2),
    (300, 248, 1032, 256, 256, 5),
])
def test_split_k(shmem, M, N, K, BM, BN, parts):
    dtype, grid = BF16, 64
    A, B, a, b = operands(shmem, M, N, K, dtype, 8)
    cg = shmem.zeros((M, N), dtype=dtype)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total,), dtype=torch.int32)
    P = shmem.zeros((grid, BM * BN), dtype=F32)
    locks = shmem.zeros((grid,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, grid, BM, BN, 64, 2, ops.EPI_ALL_SCATTER)
    kw = dict(partials=P, locks=locks, split_k=parts)
    assert "_rows" in ops.gemm_plan_name(*args, **kw)
    for launch in (1, 2):
        ops.gemm_launch(*args, **kw)
        torch.cuda.synchronize()
        check_close(cg, O.shard_gemm(A, B, dtype), f"launch {launch}")
        assert flags.cpu().tolist() == [launch] * total and not locks.any()


def test_same_sums_as_a_weight_along_k(shmem):
    """The product of a row-major B and of the same B along K: the same tile adds the same terms in the same order."""
    M, N, K, BM, BN = 512, 512, 712, 256, 256
    A, B, a, b = operands(shmem, M, N, K, BF16)
    nk = place(shmem, B.T, False, 0, 0).T
    got = []
    for w in (b, nk):
        cg = shmem.zeros((M, N), dtype=F32)
        flags = shmem.zeros((4,), dtype=torch.int32)
        ops.gemm_launch(a, w, None, cg, flags, None, 0, 1, 4, BM, BN, 64, 2, ops.EPI_ALL_SCATTER)
        torch.cuda.synchronize()
        got.append(cg.cpu())
    assert torch.equal(*got)


def test_blocks_of_the_callers_tiles(shmem):
    """256 x 64 tiles in blocks of two as 256 x 128, flags the caller's."""
    M, N, K, BM, BN, grid = 1024, 1024, 256, 256, 64, 32
    A, B, a, b = operands(shmem, M, N, K, F16)
    cg = shmem.zeros((M, N), dtype=F16)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, grid, BM, BN, 64, 4, ops.EPI_ALL_SCATTER)
    assert ops.gemm_plan_name(*args) == "256x128x64_w2x2_s3_f4_rows+two_tiles_each"
    ops.gemm_launch(*args)
    torch.cuda.synchronize()
    check_close(cg, O.shard_gemm(A, B, F16), "blocks")
    assert flags.cpu().tolist() == [1] * total


@pytest.mark.parametrize("out_dtype", [F32, F16])
@pytest.mark.parametrize("BM,BN", [(128, 128), (256, 256), (64, 64)])
def test_atomic_accumulate(shmem, out_dtype, BM, BN):
    M, N, ks, ws, dtype = 200, 136, 72, 4, F16
    A, B, a, b = operands(shmem, M, N, ks * ws, dtype)
    cg = shmem.zeros((M, N), dtype=out_dtype)
    for r in range(ws):
        args = (a[:, r * ks:(r + 1) * ks], b[r * ks:(r + 1) * ks, :], None, cg, None, None, 0, 1, 8, BM, BN, 64, 6, ops.EPI_ATOMIC_ADD)
        assert "_rows" in ops.gemm_plan_name(*args)
        ops.gemm_launch(*args)
    torch.cuda.synchronize()
    check_close(cg, O.atomics_all_reduce(O.k_shards(A, B, ws)), "sum", block_rtol=2 ** -7 if out_dtype == F32 else None)


@pytest.mark.parametrize("M,N,K,pad,shift,dtype", [
    (130, 72, 128, 4, 0, BF16),    # rows off the 16 bytes
    (130, 72, 128, 0, 4, BF16),    # the base
    (130, 76, 128, 0, 0, BF16),    # a last chunk that reaches past the row
    (130, 72, 132, 0, 0, BF16),    # A's rows
    (130, 72, 1152, 0, 0, F32),    # fp32
])
def test_what_stays_gathered(shmem, M, N, K, pad, shift, dtype):
    A, B, a, b = operands(shmem, M, N, K, dtype, pad, shift)
    cg = shmem.zeros((M, N), dtype=dtype)
    flags = shmem.zeros((6,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, 3, 64, 64, 64, 2, ops.EPI_ALL_SCATTER)
    name = ops.gemm_plan_name(*args)
    assert name.endswith("_gather") or dtype == F32 and name.endswith("_gather_fp32")
    ops.gemm_launch(*args)
    torch.cuda.synchronize()
    check_close(cg, O.shard_gemm(A, B, dtype), "gathered")


@pytest.mark.parametrize("M,N,K,BM,BN,pad,shift", [
    (1, 64, 8, 64, 64, 0, 0),         # one chunk of K, one row
    (3, 40, 72, 64, 64, 8, 0),        # N inside a cell, a block of K that holds a single chunk
    (16, 1376, 200, 64, 64, 0, 8),
    (32, 520, 1032, 64, 128, 0, 0),   # two blocks a wave in flight and one more
    (33, 328, 1024, 64, 64, 16, 0),
    (200, 504, 2056, 128, 64, 0, 0),
    (250, 120, 576, 256, 128, 24, 8),
])
@pytest.mark.parametrize("dtype,out", [(BF16, BF16), (F16, F32)])
def test_cells(shmem, M, N, K, BM, BN, pad, shift, dtype, out):
    A, B, a, b = operands(shmem, M, N, K, dtype, pad, shift)
    cg = shmem.full((M, N), 7, dtype=out)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total + 1,), dtype=torch.int32)
    locks = shmem.zeros((256,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, 256, BM, BN, 64, 2, ops.EPI_ALL_SCATTER)
    kw = dict(locks=locks, num_xcds=8)
    assert ops.gemm_plan_name(*args, **kw) == ("cells_16x32_rows" if M <= 16 else "cells_32x32_rows")
    for launch in (1, 2):
        ops.gemm_launch(*args, **kw)
        torch.cuda.synchronize()
        check_close(cg, O.shard_gemm(A, B, out), f"launch {launch}")
        assert flags.cpu().tolist() == [launch] * total + [0] and not locks.any()


@pytest.mark.parametrize("M,N,K", [(16, 256, 8200), (5, 1376, 4096)])
def test_cells_that_share_k(shmem, M, N, K):
    A, B, a, b = operands(shmem, M, N, K, BF16)
    cg = shmem.zeros((M, N), dtype=BF16)
    total = ops.cdiv(N, 64)
    flags = shmem.zeros((total,), dtype=torch.int32)
    P = shmem.zeros((256, 64 * 64), dtype=F32)
    locks = shmem.zeros((256,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, 256, 64, 64, 64, 2, ops.EPI_ALL_SCATTER)
    kw = dict(partials=P, locks=locks, num_xcds=8)
    assert ops.gemm_plan_name(*args, **kw) == ("cells_16x32_rows" if M <= 16 else "cells_32x32_rows")
    for launch in (1, 2):
        ops.gemm_launch(*args, **kw)
        torch.cuda.synchronize()
        check_close(cg, O.shard_gemm(A, B, BF16), f"launch {launch}")
        assert flags.cpu().tolist() == [launch] * total and not locks.any()


@pytest.mark.parametrize("M", [7, 13, 40])  # (8, 16 and 32 rows of A a cell)
@pytest.mark.parametrize("out_dtype", [F32, F16])
def test_cells_add_with_atomics(shmem, M, out_dtype):
    N, ks, ws = 136, 72, 4
    A, B, a, b = operands(shmem, M, N, ks * ws, F16)
    cg = shmem.zeros((M, N), dtype=out_dtype)
    for r in range(ws):
        args = (a[:, r * ks:(r + 1) * ks], b[r * ks:(r + 1) * ks, :], None, cg, None, None, 0, 1, 256, 64, 64, 64, 6, ops.EPI_ATOMIC_ADD)
        assert ops.gemm_plan_name(*args, num_xcds=8) == ("cells_16x32_rows" if M <= 16 else "cells_32x32_rows")
        ops.gemm_launch(*args, num_xcds=8)
    torch.cuda.synchronize()
    check_close(cg, O.atomics_all_reduce(O.k_shards(A, B, ws)), "sum", block_rtol=2 ** -7 if out_dtype == F32 else None)
