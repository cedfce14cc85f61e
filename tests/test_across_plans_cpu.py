"""Launches whose tiles need not divide the caller's: which calls are planned so, and what is planned around them."""

import ctypes
import random

import pytest

from iris_amd import _native, ops
from test_gemm_plans_cpu import BF16, F32, plan, plan_args

F16 = 1


def one_shot(M, N, K, BM, BN, dtype, ws, phase, partial, **kw):
    return plan(M, N, K, BM, BN, dtype, ws, epilogue=ops.EPI_ONE_SHOT, phase=phase, c=9 << 32, c_dtype=partial, stride_cm=N, stride_cn=1,
                stride_cm_global=N, **kw)[0]


@pytest.mark.parametrize("M,N,K,BM,BN,dtype,ws,partial,inside", [
    # more of the caller's tiles than programs: never inside, in however few tiles the producer runs
    (1219, 1016, 1168, 64, 64, BF16, 2, BF16, False), (1219, 1016, 1168, 64, 64, BF16, 8, BF16, False),
    (1911, 2120, 472, 128, 64, BF16, 8, BF16, False), (1330, 3560, 552, 64, 128, BF16, 4, BF16, False),
    # one round of large ones
    (2550, 2376, 344, 256, 256, BF16, 8, BF16, False), (418, 760, 256, 128, 128, F32, 2, F32, False),
    # ... and of small ones
    (748, 1504, 256, 128, 64, F32, 4, F32, True), (580, 2880, 227, 128, 64, BF16, 4, BF16, True),
])
def test_the_reduce_of_a_producer_in_other_tiles(M, N, K, BM, BN, dtype, ws, partial, inside):
    rows = dict(stride_bk=N, stride_bn=1) if K == 227 else {}
    assert "+across_the_tiles" in one_shot(M, N, K, BM, BN, dtype, ws, ops.PHASE_TWO_KERNELS, partial, **rows)
    name = one_shot(M, N, K, BM, BN, dtype, ws, ops.PHASE_FUSED, partial, **rows)
    assert name.endswith("+reduce") and name.endswith("+across_the_tiles+kernel+reduce") != inside


@pytest.mark.parametrize("M,N,K,BM,BN,dtype", [(16, 4096, 1376, 64, 64, BF16), (46, 128, 22784, 64, 64, F16), (53, 1344, 1008, 128, 128, F32)])
def test_the_few_rows_kernel_by_name_is_no_program_that_also_reduces(M, N, K, BM, BN, dtype):
    """IRIS_PHASE_FUSED with IRIS_GEMM_VARIANT_FEW_ROWS is refused, whatever the launcher itself would choose for the call."""
    args = plan_args(M, N, K, BM, BN, dtype, 4, epilogue=ops.EPI_ONE_SHOT, phase=ops.PHASE_FUSED, c=9 << 32, c_dtype=dtype, stride_cm=N,
                     stride_cn=1, stride_cm_global=N, variant=ops.VARIANT_FEW_ROWS)
    name = ctypes.create_string_buffer(256)
    assert _native.lib().iris_gemm_plan_name(ctypes.byref(args), name, 256) == _native.HIP_ERROR_INVALID_VALUE
    args.phase = ops.PHASE_TWO_KERNELS
    assert _native.lib().iris_gemm_plan_name(ctypes.byref(args), name, 256) == 0 and name.value.startswith(b"few_rows")


@pytest.mark.parametrize("M,N,K,BM,BN,kw", [
    (1764, 940, 401, 256, 64, dict(epilogue=ops.EPI_ATOMIC_ADD, stride_cm_global=940)),
    (2000, 829, 349, 256, 128, dict(epilogue=ops.EPI_ATOMIC_ADD, stride_cm_global=829, stride_bk=829, stride_bn=1, partials=0, locks=0)),
    (5197, 322, 320, 128, 128, dict(epilogue=ops.EPI_ONE_SHOT, phase=ops.PHASE_PRODUCE, c=9 << 32, stride_cm=322, stride_cn=1, stride_bk=322,
                                    stride_bn=1, partials=0, locks=0)),
])
def test_operands_that_are_gathered_are_not_left_to_the_loader_of_single_elements(M, N, K, BM, BN, kw):
    """There is no gathering 64 x 64 tile for fp32 of a short K."""
    assert "_gather" in plan(M, N, K, BM, BN, F32, **kw)[0]


def test_no_tile_that_loads_single_elements_for_one_that_does_not():
    rng, seen = random.Random(5), 0
    for _ in range(6000):
        M, N, K = (int(2 ** rng.uniform(0, 13)) for _ in range(3))
        BM, BN = rng.choice([(64, 64), (128, 128), (256, 64), (256, 128)])
        kw = rng.choice([dict(epilogue=ops.EPI_ATOMIC_ADD, stride_cm_global=N), dict(),
                         dict(epilogue=ops.EPI_ONE_SHOT, phase=ops.PHASE_PRODUCE, c=9 << 32, stride_cm=N, stride_cn=1)])
        if rng.random() < 0.6:
            kw = dict(kw, stride_bk=N, stride_bn=1)
        own = plan(M, N, K, BM, BN, F32, variant=ops.VARIANT_PERSISTENT, **kw)[0]
        if "generic" not in own:
            assert "generic" not in plan(M, N, K, BM, BN, F32, **kw)[0], (M, N, K, BM, BN, kw, own)
            seen += "_gather" in own
    assert seen > 100


@pytest.mark.parametrize("M,N,K,dtype,kw", [
    (966, 992, 2288, F16, {}), (108, 5288, 1505, BF16, {}),
    (59, 7648, 488, BF16, dict(epilogue=ops.EPI_ATOMIC_ADD, stride_cm_global=7648)),
])
def test_a_word_counts_the_parts_of_a_large_tile(M, N, K, dtype, kw):
    """Parts of the caller's tiles count in a word each, so that a tile may have any number of them."""
    assert plan(M, N, K, 1024, 1024, dtype, **kw)[0].startswith("64x64") and "+parts_of_tiles" in plan(M, N, K, 1024, 1024, dtype, **kw)[0]


@pytest.mark.parametrize("M,N,K,BM,BN,dtype,ws,kw,want", [
    # parts that hand over, to four and eight copies
    (39, 287, 3816, 128, 128, F32, 8, dict(stride_bk=287, stride_bn=1), ("64x64x64_w2x2_gather_fp32+parts_of_tiles", 16)),
    (92, 192, 28736, 256, 64, BF16, 8, dict(stride_bk=192, stride_bn=1), ("64x64x128_w2x2_s4_f4_rows+parts_of_tiles", 16)),
    (895, 671, 2685, 64, 64, F32, 4, dict(stride_bk=671, stride_bn=1), ("64x64x64_w2x2_gather_fp32", 1)),
    # a last round whose K is shared out
    (4035, 1145, 18287, 128, 128, BF16, 4, dict(c_global_dtype=BF16), ("128x128x64_w2x2_s4_f4_gather_dma+last_round_in_8_parts", 1)),
    # ... and what other tiles and parts that add their own sums are for
    (828, 2688, 20672, 256, 64, BF16, 1, {}, ("128x256x64_w1x4_s3_f4", 3)),
    (4088, 131, 35880, 64, 128, F16, 4, {}, ("128x128x64_w2x2_s4_f4", 4)),
    (1104, 1126, 11095, 64, 64, BF16, 1, {}, ("128x128x64_w2x2_s4_f4_gather_dma", 3)),
])
def test_atomics(M, N, K, BM, BN, dtype, ws, kw, want):
    assert plan(M, N, K, BM, BN, dtype, ws, **dict(dict(epilogue=ops.EPI_ATOMIC_ADD, c_global_dtype=F32, stride_cm_global=N), **kw)) == want


@pytest.mark.parametrize("kw", [dict(mm_begin_timestamp=10 << 32, mm_end_timestamp=11 << 32), dict(mm_end_timestamp=11 << 32), dict(split_k=1),
                                dict(split_k=2), dict(variant=ops.VARIANT_PERSISTENT), dict(num_sms=248)])
def test_what_is_asked_for_keeps_the_callers_tiles(kw):
    """Timestamps are the caller's tiles' own; parts, a variant and fewer programs than CUs are the caller's choice."""
    atomics = dict(epilogue=ops.EPI_ATOMIC_ADD, c_global_dtype=F32, stride_cm_global=1296)
    assert plan(965, 1296, 4504, 128, 128, F16, **atomics)[0].startswith("256x64x64")
    assert plan(965, 1296, 4504, 128, 128, F16, **dict(atomics, **kw))[0].startswith("128x128x64")
    assert "+across_the_tiles" in plan(1911, 2120, 472, 256, 64)[0]
    if kw.get("split_k") != 2:  # (the caller's tiles are more than half the programs: no two parts of them)
        assert "across" not in plan(1911, 2120, 472, 256, 64, **kw)[0]


@pytest.mark.parametrize("M,N,K,BM,BN,dtype,ws,across", [
    # one or two K-steps, in the caller's tiles and in blocks of them
    (1034, 2135, 64, 64, 128, F16, 8, False), (2654, 1920, 128, 256, 256, F16, 8, False), (290, 5765, 64, 128, 64, BF16, 8, True),
    # rows of an odd length, to eight copies and to one
    (6500, 679, 320, 64, 128, BF16, 8, False), (2011, 2523, 186, 64, 128, BF16, 1, False), (1911, 2121, 472, 256, 64, BF16, 1, True),
    (1911, 2120, 472, 256, 64, BF16, 8, True),
])
def test_where_the_stores_are_most_of_it(M, N, K, BM, BN, dtype, ws, across):
    row = K + 1 if K == 186 else K
    assert ("+across_the_tiles" in plan(M, N, K, BM, BN, dtype, ws, row=row)[0]) == across
