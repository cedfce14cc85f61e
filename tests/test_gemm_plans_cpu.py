"""Which kernel the launcher plans for small products, on both sides of every line where the faster one changes
(``iris_gemm_plan_name`` reads the arguments only: no GPU, and the pointers below are never followed)."""

import ctypes

import pytest

from iris_amd import _native, ops

BF16, F32 = 2, 0


def plan_args(M, N, K, BM, BN, dtype=BF16, ws=1, base=1 << 32, row=None, **kw):
    args = _native.GemmArgs()
    args.a, args.b, args.c_global = base, 2 << 32, 4 << 32
    args.tile_completed, args.heap_bases = 5 << 32, 6 << 32
    args.partials, args.locks, args.partials_slot_elems = 7 << 32, 8 << 32, BM * BN
    args.M, args.N, args.K = M, N, K
    args.stride_am, args.stride_ak, args.stride_bk, args.stride_bn = row or K, 1, 1, row or K
    args.stride_cm_global, args.stride_cn_global = N * ws, 1
    args.block_m, args.block_n, args.block_k, args.group_size_m = BM, BN, 64, 4
    args.num_sms, args.num_xcds, args.world_size = 256, 8, ws
    args.ab_dtype = args.c_dtype = args.c_global_dtype = dtype
    args.epilogue, args.notify = ops.EPI_ALL_SCATTER, 1
    for name, value in kw.items():
        setattr(args, name, value)
    return args


def plan(*args, **kw):
    args, lib = plan_args(*args, **kw), _native.lib()
    name, parts = ctypes.create_string_buffer(256), ctypes.c_int(0)
    assert lib.iris_gemm_plan_name(ctypes.byref(args), name, 256) == 0
    assert lib.iris_gemm_split_k(ctypes.byref(args), ctypes.byref(parts)) == 0
    return name.value.decode(), parts.value


PARTS = "64x64x128_w2x2_s4_f4+parts_of_tiles"


@pytest.mark.parametrize("M,N,K,BM,BN,want", [
    # a row-major weight: cells up to a K whose half lines no longer come in time, and for what 32 rows of them share
    (1, 1376, 4096, 64, 64, ("cells_16x32_rows", 1)),
    (16, 1376, 4096, 64, 64, ("cells_16x32_rows", 1)), (17, 1376, 4096, 64, 64, ("cells_32x32_rows", 1)),
    (27, 256, 28032, 256, 64, ("cells_32x32_rows", 1)),
    (128, 1376, 4096, 64, 64, ("cells_32x32_rows", 1)),
    (28, 4864, 7936, 64, 64, ("64x64x128_w2x2_s4_f4_rows", 3)),
    (138, 128, 32000, 64, 64, ("64x64x128_w2x2_s4_f4_rows", 16)),
    # rows off the 16 bytes
    (16, 1380, 1024, 64, 64, ("64x64x128_w2x2_gather", 4)),
])
def test_row_major_weights(M, N, K, BM, BN, want):
    assert plan(M, N, K, BM, BN, stride_bk=N, stride_bn=1) == want


@pytest.mark.parametrize("M,N,BM,BN,K,want", [
    # 32 tiles of 128 x 128 and the like: parts fill the chip, a long K is shared out instead
    (256, 2048, 128, 128, 512, (PARTS, 1)),
    (256, 2048, 128, 128, 2048, (PARTS, 1)),
    (256, 2048, 128, 128, 16384, ("128x128x64_w2x2_s4_f4", 8)),
    (256, 2048, 128, 128, 36864, ("128x128x64_w2x2_s4_f4", 8)),
    (256, 2048, 256, 64, 2048, (PARTS, 1)),
    (256, 2048, 256, 64, 36864, ("256x64x64_w4x1_s3_f4", 8)),
    (256, 2048, 256, 128, 2048, (PARTS, 1)),
    (256, 2048, 256, 128, 36864, ("256x128x64_w2x2_s3_f4", 16)),
    (256, 2048, 256, 256, 2048, (PARTS, 1)),
    (256, 2048, 256, 256, 36864, ("256x256x64_w2x4_s2", 16)),
    (256, 2048, 64, 64, 36864, ("64x64x128_w2x2_s4_f4", 2)),
    # 256 cells of 32 x 32
    (512, 512, 64, 64, 2048, ("cells_32x32", 1)),
    (512, 512, 64, 64, 36864, ("64x64x128_w2x2_s4_f4", 4)),
    (512, 512, 128, 128, 8192, ("cells_32x32", 1)),
    (512, 512, 128, 128, 36864, ("128x128x64_w2x2_s4_f4", 16)),
    (512, 512, 256, 64, 36864, ("256x64x64_w4x1_s3_f4", 16)),
    (512, 512, 256, 128, 36864, ("256x128x64_w2x2_s3_f4", 16)),
    (512, 512, 256, 256, 36864, (PARTS, 3)),
    # a batch too tall for the few-rows kernel
    (128, 1376, 64, 64, 4096, ("cells_32x32", 1)),
    (128, 1376, 128, 128, 36864, ("128x128x64_w2x2_s4_f4", 16)),
])
def test_small_products(M, N, BM, BN, K, want):
    assert plan(M, N, K, BM, BN) == want


@pytest.mark.parametrize("M,N,K,few", [
    (17, 4096, 21136, True), (32, 4096, 16384, True), (24, 4096, 21136, True), (32, 4096, 21136, False),
    (32, 1376, 21136, True), (17, 4776, 4096, True), (17, 4776, 8192, False), (32, 8192, 36864, False),
    (16, 8192, 36864, True),
])
def test_rows_of_a_long_k(M, N, K, few):
    assert plan(M, N, K, 64, 64)[0].startswith("few_rows") == few
    # ... asked for by name, the kernel still takes them
    assert plan(M, N, K, 64, 64, variant=ops.VARIANT_FEW_ROWS)[0].startswith("few_rows")


def test_rows_off_the_cache_lines():
    # a shard of a wider operand whose rows do not start on cache lines, by their stride or by the first of them
    assert plan(32, 8192, 1024 * 16, 64, 64, row=1 << 17) == plan(32, 8192, 1024 * 16, 64, 64)
    on, off = plan(32, 4096, 20480, 64, 64, row=1 << 16)[0], plan(32, 4096, 20480, 64, 64, row=1 << 16, base=(1 << 32) + 32)[0]
    assert on.startswith("few_rows") and not off.startswith("few_rows")


def test_no_split_asked_for_stays_unsplit():
    for K in (512, 36864):
        assert plan(512, 512, K, 128, 128, split_k=1)[1] == 1
        assert plan(256, 2048, K, 128, 128, split_k=1) == ("128x128x64_w2x2_s4_f4", 1)


def test_fp32():
    assert plan(512, 512, 512, 128, 128, dtype=F32)[0] == "cells_32x32"
    name, parts = plan(512, 512, 36864, 128, 128, dtype=F32)
    assert name == "128x128x32_w2x2_s4_f4_fp32" and parts == 16


@pytest.mark.parametrize("M,N,K,BM,BN,ws,partial,inside", [
    (64, 640, 320, 256, 64, 2, F32, True), (64, 640, 1376, 256, 64, 2, F32, False),
    (64, 4096, 640, 256, 64, 8, BF16, True),
    (128, 4096, 128, 256, 64, 8, F32, True), (128, 320, 128, 256, 64, 8, F32, False),  # 64 tiles, and 5
    (2000, 640, 320, 256, 64, 2, F32, True), (2000, 640, 320, 256, 64, 8, F32, False),
    (16, 4096, 128, 64, 64, 2, F32, True), (16, 4096, 320, 64, 64, 2, F32, False), (1, 320, 128, 256, 128, 2, F32, False),
    (1999, 4096, 1376, 256, 128, 8, BF16, False), (785, 2752, 216, 256, 64, 8, F32, True),
])
def test_the_reduce_inside_the_program_or_behind_it(M, N, K, BM, BN, ws, partial, inside):
    name, _ = plan(M, N, K, BM, BN, ws=ws, epilogue=ops.EPI_ONE_SHOT, phase=ops.PHASE_FUSED, c=3 << 32, c_dtype=partial,
                   stride_cm=N, stride_cn=1, stride_cm_global=N)
    assert name.endswith("+reduce") and name.endswith("+kernel+reduce") != inside


@pytest.mark.parametrize("M,N,K,BM,BN,ws,rows,inside", [
    # a row-major weight, whose producer is faster than the program that also reduces
    (1000, 1024, 1024, 64, 64, 8, True, True), (1000, 1024, 1504, 64, 64, 8, True, False),
    (16, 4096, 256, 64, 64, 8, True, True), (16, 4096, 1376, 64, 64, 8, True, False),
    (2048, 2048, 392, 128, 128, 2, True, True), (2048, 2048, 1288, 128, 128, 2, True, False),
    (2048, 2048, 392, 128, 128, 8, True, False),
    (4096, 2048, 136, 256, 128, 2, True, True), (4096, 2048, 392, 256, 128, 2, True, False),
    # rows along K off the 16 bytes
    (16, 4096, 133, 64, 64, 8, False, True), (16, 4096, 637, 64, 64, 8, False, False),
    (2048, 2048, 573, 128, 128, 2, False, True), (2048, 2048, 1285, 128, 128, 2, False, False),
    (4096, 1024, 389, 256, 64, 8, False, False), (1000, 1024, 1501, 64, 64, 8, False, True),
])
def test_where_operands_that_are_gathered_inside_are_reduced(M, N, K, BM, BN, ws, rows, inside):
    kw = dict(stride_bk=N, stride_bn=1) if rows else {}
    name, _ = plan(M, N, K, BM, BN, ws=ws, epilogue=ops.EPI_ONE_SHOT, phase=ops.PHASE_FUSED, c=9 << 32, stride_cm=N, stride_cn=1,
                   stride_cm_global=N, **kw)
    assert name.endswith("+kernel+reduce") != inside, name


@pytest.mark.parametrize("M,N,K,BM,BN", [(828, 2688, 20672, 256, 64), (2023, 192, 22656, 256, 128)])
def test_atomics_to_other_gpus_add_whole_sums(M, N, K, BM, BN):
    """Parts of K that each add their own sums would send all of them over the links; ranks of one GPU take them.  (Without
    a workspace K is not shared out in any other way.)"""
    kw = dict(epilogue=ops.EPI_ATOMIC_ADD, c_global_dtype=F32, ws=2, partials=0, locks=0)
    assert plan(M, N, K, BM, BN, **kw)[1] > 1
    assert plan(M, N, K, BM, BN, scope=ops.SCOPE_SYSTEM, **kw)[1] == 1
