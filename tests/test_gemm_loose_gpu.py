"""The LDS-DMA tiles for operands along K at any alignment (``_gather_dma``): every tile's edges, a K that cuts each chunk of
a step, in the first, a middle and the only step of a tile or of a part, bases and rows 2 to 14 bytes off, NaN around the
operands and infinities in what a cut chunk repeats, against the CPU oracle."""

import pytest
import torch

from iris_amd import ops
from oracle import iris_oracle as O
from parity import check_close, make_ab
from test_gemm_gather_gpu import place

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def operands(shmem, M, N, K, dtype, pad, shift):
    A, B = make_ab(M, N, K, dtype)
    return A, B, place(shmem, A, False, pad, shift), place(shmem, B.T, False, pad, shift).T


@pytest.mark.parametrize("M,N,K,BM,BN,pad,shift,name", [
    (130, 70, 8, 64, 64, 1, 3, "64x64x128_w2x2_s4"),          # one chunk
    (130, 70, 9, 64, 64, 0, 0, "64x64x128_w2x2_s4"),          # the second holds one k
    (130, 70, 127, 64, 64, 0, 0, "64x64x128_w2x2_s4"),        # the only step, cut in its last chunk
    (130, 70, 128, 64, 64, 4, 0, "64x64x128_w2x2_s4"),        # whole steps, rows 8 bytes off
    (90, 201, 129, 64, 64, 0, 1, "64x64x128_w2x2_s4"),        # the last step is one k, moved back into the step before
    (90, 201, 1500, 64, 64, 0, 0, "64x64x128_w2x2_s4"),
    (257, 75, 1031, 128, 64, 2, 2, "128x64x64_w2x2_s4"),
    (40, 260, 203, 64, 128, 1, 0, "64x128x64_w2x2_s4"),
    (300, 136, 642, 128, 128, 5, 0, "128x128x64_w2x2_s4"),
    (520, 72, 449, 256, 64, 0, 7, "256x64x64_w4x1_s3"),
    (300, 200, 577, 256, 128, 2, 5, "256x128x64_w2x2_s3"),
    (300, 200, 61, 256, 128, 0, 0, "256x128x64_w2x2_s3"),
    (513, 300, 202, 256, 256, 0, 6, "256x256x64_w2x4_s2"),
    (300, 520, 1101, 256, 256, 3, 0, "256x256x64_w2x4_s2"),
    (300, 520, 65, 256, 256, 0, 0, "256x256x64_w2x4_s2"),     # two steps
])
@pytest.mark.parametrize("dtype,out", [(BF16, BF16), (F16, F16), (BF16, F32)])
def test_scatter(shmem, M, N, K, BM, BN, pad, shift, name, dtype, out):
    A, B, a, b = operands(shmem, M, N, K, dtype, pad, shift)
    cg = shmem.full((M, N), 7, dtype=out)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total + 1,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, 3, BM, BN, 64, 2, ops.EPI_ALL_SCATTER)
    plan = ops.gemm_plan_name(*args, variant=ops.VARIANT_PERSISTENT)
    assert plan.startswith(name) and plan.endswith("_gather_dma"), plan
    for launch in (1, 2):
        ops.gemm_launch(*args, variant=ops.VARIANT_PERSISTENT)
        torch.cuda.synchronize()
        check_close(cg, O.shard_gemm(A, B, out), f"launch {launch}")
        assert flags.cpu().tolist() == [launch] * total + [0]


@pytest.mark.parametrize("cut", range(1, 8))
@pytest.mark.parametrize("chunk", [0, 3, 4, 7])
def test_every_cut_of_a_step(shmem, cut, chunk):
    """K = two whole steps of 64, some chunks and `cut` more: the same sums as with the operands' last rows zero-padded."""
    M, N, K = 130, 130, 128 + 8 * chunk + cut
    A, B, a, b = operands(shmem, M, N, K, BF16, 0, 0)
    cg = shmem.zeros((M, N), dtype=F32)
    flags = shmem.zeros((4,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, 4, 128, 128, 64, 2, ops.EPI_ALL_SCATTER)
    assert ops.gemm_plan_name(*args, variant=ops.VARIANT_PERSISTENT) == "128x128x64_w2x2_s4_f4_gather_dma"
    ops.gemm_launch(*args, variant=ops.VARIANT_PERSISTENT)
    pad = 8 - cut
    ap, bp = shmem.zeros((M, K + pad), dtype=BF16), shmem.zeros((N, K + pad), dtype=BF16)
    ap[:, :K], bp[:, :K] = a, b.T
    whole = shmem.zeros((M, N), dtype=F32)
    ops.gemm_launch(ap, bp.T, None, whole, flags, None, 0, 1, 4, 128, 128, 64, 2, ops.EPI_ALL_SCATTER,
                    variant=ops.VARIANT_PERSISTENT)
    torch.cuda.synchronize()
    # the moved chunk's k stand at other places of the last MFMA, whose own order of addition is not the rows': a few ulps
    assert torch.allclose(cg, whole, rtol=1e-5, atol=1e-5)


def test_infinities_are_met_once(shmem):
    """An infinity in the k that a cut chunk repeats: an infinite result, not a NaN."""
    M, N, K = 64, 64, 131
    A, B, a, b = operands(shmem, M, N, K, BF16, 0, 0)
    a[3, 126], b[126, 5] = float("inf"), 1.0
    b[127, 9], a[7, 127] = float("inf"), 0.5
    cg = shmem.zeros((M, N), dtype=F32)
    flags = shmem.zeros((1,), dtype=torch.int32)
    ops.gemm_launch(a, b, None, cg, flags, None, 0, 1, 1, 64, 64, 64, 2, ops.EPI_ALL_SCATTER, variant=ops.VARIANT_PERSISTENT)
    torch.cuda.synchronize()
    want = a.float().cpu() @ b.float().cpu()
    assert torch.equal(torch.isnan(cg.cpu()), torch.isnan(want)) and torch.equal(torch.isinf(cg.cpu()), torch.isinf(want))


@pytest.mark.parametrize("M,N,K,BM,BN,parts", [
    (100, 200, 1030, 64, 64, 3),     # the owner's hand-over
    (100, 200, 1030, 64, 64, 8),     # sliced: the last part is the cut step
    (256, 136, 1023, 128, 128, 4),
    (200, 72, 779, 256, 64, 4),
    (300, 250, 1025, 256, 128, 2),   # the pair hand-over
    (300, 250, 1025, 256, 256, 2),
    (300, 250, 1025, 256, 256, 5),
])
def test_split_k(shmem, M, N, K, BM, BN, parts):
    dtype, grid = BF16, 64
    A, B, a, b = operands(shmem, M, N, K, dtype, 1, 0)
    cg = shmem.zeros((M, N), dtype=dtype)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total,), dtype=torch.int32)
    P = shmem.zeros((grid, BM * BN), dtype=F32)
    locks = shmem.zeros((grid,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, grid, BM, BN, 64, 2, ops.EPI_ALL_SCATTER)
    kw = dict(partials=P, locks=locks, split_k=parts)
    assert "_gather_dma" in ops.gemm_plan_name(*args, **kw)
    for launch in (1, 2):
        ops.gemm_launch(*args, **kw)
        torch.cuda.synchronize()
        check_close(cg, O.shard_gemm(A, B, dtype), f"launch {launch}")
        assert flags.cpu().tolist() == [launch] * total and not locks.any()


@pytest.mark.parametrize("out_dtype", [F32, F16])
@pytest.mark.parametrize("BM,BN", [(128, 128), (256, 256), (64, 64)])
def test_atomic_accumulate(shmem, out_dtype, BM, BN):
    M, N, ks, ws, dtype = 200, 136, 67, 4, F16
    A, B, a, b = operands(shmem, M, N, ks * ws, dtype, 1, 1)
    cg = shmem.zeros((M, N), dtype=out_dtype)
    for r in range(ws):
        args = (a[:, r * ks:(r + 1) * ks], b[r * ks:(r + 1) * ks, :], None, cg, None, None, 0, 1, 8, BM, BN, 64, 6, ops.EPI_ATOMIC_ADD)
        assert "_gather_dma" in ops.gemm_plan_name(*args)
        ops.gemm_launch(*args)
    torch.cuda.synchronize()
    check_close(cg, O.atomics_all_reduce(O.k_shards(A, B, ws)), "sum", block_rtol=2 ** -7 if out_dtype == F32 else None)


def test_blocks_of_the_callers_tiles(shmem):
    M, N, K, BM, BN, grid = 1024, 1024, 259, 256, 64, 32
    A, B, a, b = operands(shmem, M, N, K, F16, 0, 0)
    cg = shmem.zeros((M, N), dtype=F16)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, grid, BM, BN, 64, 4, ops.EPI_ALL_SCATTER)
    assert ops.gemm_plan_name(*args) == "256x128x64_w2x2_s3_f4_gather_dma+two_tiles_each"
    ops.gemm_launch(*args)
    torch.cuda.synchronize()
    check_close(cg, O.shard_gemm(A, B, F16), "blocks")
    assert flags.cpu().tolist() == [1] * total


@pytest.mark.parametrize("M,N,K,lda,dtype", [
    (130, 70, 7, 7, BF16),        # K shorter than a chunk: element by element
    (130, 70, 1030, 1030, F32),   # fp32
    (64, 70, 128, 100, BF16),     # rows of A that overlap
])
def test_what_stays_as_it_was(shmem, M, N, K, lda, dtype):
    A, B = make_ab(M, N, K, dtype)
    flat = shmem.zeros((M * lda + K + 64,), dtype=dtype)
    a = flat[1:].as_strided((M, K), (lda, 1))
    a.copy_(A) if lda >= K else flat.copy_(torch.randn(flat.shape, generator=torch.Generator().manual_seed(5)).to(dtype) * 0.1)
    A = a.cpu()
    b = place(shmem, B.T, False, 1, 0).T
    cg = shmem.zeros((M, N), dtype=dtype)
    flags = shmem.zeros((8,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, 3, 64, 64, 64, 2, ops.EPI_ALL_SCATTER)
    assert "_gather_dma" not in ops.gemm_plan_name(*args)
    ops.gemm_launch(*args)
    torch.cuda.synchronize()
    check_close(cg, O.shard_gemm(A, B, dtype), "as it was")


@pytest.mark.parametrize("M,N,K,BM,BN,pad,shift,kernel", [
    (1, 300, 4099, 64, 64, 0, 0, "few_rows_16xN"),     # one k in the last chunk
    (3, 50, 9, 64, 64, 0, 1, "few_rows_16xN"),         # two chunks, N no multiple of a workgroup's columns
    (8, 72, 8, 64, 64, 1, 0, "few_rows_16xN"),         # one whole chunk off the 16 bytes
    (9, 200, 1407, 64, 64, 3, 5, "few_rows_16xN"),
    (17, 130, 2111, 64, 64, 0, 0, "few_rows_16xN"),
    (30, 201, 63, 64, 128, 0, 0, "few_rows_16xN"),     # one block of K, cut in its last chunk
    (20, 4200, 2050, 64, 64, 0, 0, "few_rows_32xN"),   # blocks of 32 rows
    (50, 272, 3001, 64, 64, 1, 0, "few_rows_32xN"),
    (4, 192, 8197, 64, 64, 0, 0, "few_rows_16xN"),     # K shared out over workgroups
    (130, 330, 1021, 64, 64, 0, 3, "cells_32x32"),
    (200, 500, 515, 128, 64, 0, 0, "cells_32x32"),
])
@pytest.mark.parametrize("dtype,out", [(BF16, BF16), (F16, F32)])
def test_few_rows_and_cells(shmem, M, N, K, BM, BN, pad, shift, kernel, dtype, out):
    A, B, a, b = operands(shmem, M, N, K, dtype, pad, shift)
    cg = shmem.full((M, N), 7, dtype=out)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total + 1,), dtype=torch.int32)
    P = shmem.zeros((256, BM * BN), dtype=F32)
    locks = shmem.zeros((256,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, 256, BM, BN, 64, 2, ops.EPI_ALL_SCATTER)
    kw = dict(partials=P, locks=locks, num_xcds=8)
    assert ops.gemm_plan_name(*args, **kw) == kernel + "_gather_dma"
    for launch in (1, 2):
        ops.gemm_launch(*args, **kw)
        torch.cuda.synchronize()
        check_close(cg, O.shard_gemm(A, B, out), f"launch {launch}")
        assert flags.cpu().tolist() == [launch] * total + [0] and not locks.any()


@pytest.mark.parametrize("M,N,K,name", [(5, 70, 1031, "few_rows_16xN_gather_dma"), (70, 130, 517, "few_rows_32xN_gather_dma")])
def test_fp32_few_rows(shmem, M, N, K, name):
    A, B, a, b = operands(shmem, M, N, K, F32, 1, 1)
    cg = shmem.zeros((M, N), dtype=F32)
    flags = shmem.zeros((16,), dtype=torch.int32)
    locks = shmem.zeros((256,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, 256, 64, 64, 64, 2, ops.EPI_ALL_SCATTER)
    assert ops.gemm_plan_name(*args, locks=locks, num_xcds=8) == name
    ops.gemm_launch(*args, locks=locks, num_xcds=8)
    torch.cuda.synchronize()
    check_close(cg, O.shard_gemm(A, B, F32), "fp32", block_rtol=1e-5)


def test_the_few_rows_kernel_is_not_to_be_had_for_them_by_name(shmem):
    A, B, a, b = operands(shmem, 4, 64, 131, BF16, 0, 0)
    cg = shmem.zeros((4, 64), dtype=BF16)
    flags = shmem.zeros((1,), dtype=torch.int32)
    with pytest.raises(ValueError):
        ops.gemm_plan_name(a, b, None, cg, flags, None, 0, 1, 256, 64, 64, 64, 2, ops.EPI_ALL_SCATTER,
                           variant=ops.VARIANT_FEW_ROWS)
