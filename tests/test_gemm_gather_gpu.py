"""The gathering tiles: operands that lie across K (a column-major A, a row-major B whose
rows start anywhere), and fp32 ones, against the CPU oracle; and beside them what does not come to these tiles any more,
16-bit operands along K whose rows start anywhere (odd strides, a K that is no multiple of 8, unaligned bases).  Edges in all
three directions, single and odd numbers of K-steps, split K, the three epilogues, and what stays element by element."""

import pytest
import torch

from iris_amd import ops
from oracle import iris_oracle as O
from parity import check_close, make_ab

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def place(shmem, t, across, pad, shift):
    """A device copy of host matrix ``t`` with its rows' length padded by
    ``pad`` and its base moved by ``shift`` elements; ``across``: stored
    transposed.  The memory around it is NaN: nothing outside may reach a
    result."""
    src = t.T if across else t
    rows, cols = src.shape
    flat = shmem.full((shift + rows * (cols + pad) + 64,), float("nan"), dtype=t.dtype)
    view = flat[shift:].as_strided((rows, cols), (cols + pad, 1))
    view.copy_(src)
    return view.T if across else view


CASES = [
    # M, N, K, BLK_M, BLK_N, a across, b across, pad, shift, the kernel in 16 bits and in fp32
    (130, 72, 100, 64, 64, False, False, 0, 0, "64x64x128_w2x2_s4_f4_gather_dma", "64x64x32_w2x2_s4_fp32"),  # K no multiple of 8
    (130, 70, 8, 64, 64, False, False, 1, 3, "64x64x128_w2x2_s4_f4_gather_dma", "64x64x16_w2x2_generic_fp32"),  # one chunk of K
    (96, 80, 64, 64, 64, True, True, 0, 0, "64x64x128_w2x2_gather", "64x64x16_w2x2_generic_fp32"),  # both across, whole steps
    (100, 75, 129, 64, 64, True, True, 3, 1, "64x64x128_w2x2_gather", "64x64x16_w2x2_generic_fp32"),  # ... odd in every direction
    (64, 200, 300, 64, 64, False, True, 0, 0, "64x64x128_w2x2_gather", "64x64x16_w2x2_generic_fp32"),
    (8, 8, 8, 64, 64, True, True, 0, 0, "64x64x128_w2x2_gather", "64x64x16_w2x2_generic_fp32"),  # the smallest blocks
    (300, 136, 640, 128, 128, False, True, 5, 0, "128x128x64_w2x2_gather", "128x128x32_w2x2_gather_fp32"),  # 128 x 128, two tiles a program
    (257, 129, 65, 128, 128, True, False, 1, 1, "128x128x64_w2x2_gather", "64x64x16_w2x2_generic_fp32"),  # two K-steps, the second with one k
    (40, 260, 200, 64, 128, False, True, 1, 0, "64x128x64_w2x2_gather", "64x64x16_w2x2_generic_fp32"),
    (520, 72, 449, 256, 64, False, True, 0, 7, "256x64x64_w4x1_gather", "256x64x32_w4x1_gather_fp32"),  # eight K-steps, the last with one k
    (300, 200, 577, 256, 128, True, True, 0, 0, "256x128x64_w2x2_gather", "128x128x32_w2x2_gather_fp32"),  # ten K-steps
    (300, 200, 577, 256, 128, False, False, 2, 5, "256x128x64_w2x2_s3_f4_gather_dma", "128x128x32_w2x2_gather_fp32"),
    (513, 300, 200, 256, 256, False, True, 0, 0, "256x128x64_w2x2_gather", "64x64x16_w2x2_generic_fp32"),  # several compute tiles a logical tile
    (96, 72, 40, 32, 24, False, True, 0, 0, "64x64x128_w2x2_gather", "64x64x16_w2x2_generic_fp32"),  # logical tile smaller than any compute tile
    (1, 300, 4099, 64, 64, False, True, 0, 0, "64x64x128_w2x2_gather", "64x64x64_w2x2_gather_fp32"),  # one row
    (7, 40, 72, 64, 64, True, False, 0, 0, "64x64x32_w2x2_generic", "64x64x16_w2x2_generic_fp32"),  # too few rows for a block: element by element
]


@pytest.mark.parametrize("M,N,K,BM,BN,aa,ba,pad,shift,name16,name32", CASES)
@pytest.mark.parametrize("dtype", [BF16, F16, F32])
def test_scatter(shmem, M, N, K, BM, BN, aa, ba, pad, shift, name16, name32, dtype):
    A, B = make_ab(M, N, K, dtype)
    a = place(shmem, A, aa, pad, shift)
    b = place(shmem, B, False, pad, shift) if ba else place(shmem, B.T, False, pad, shift).T
    cg = shmem.full((M, N), 7, dtype=dtype)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total + 1,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, 3, BM, BN, 64, 2, ops.EPI_ALL_SCATTER)
    assert ops.gemm_plan_name(*args) == (name32 if dtype == F32 else name16)
    for launch in (1, 2):
        ops.gemm_launch(*args)
        torch.cuda.synchronize()
        check_close(cg, O.shard_gemm(A, B, dtype), f"launch {launch}")
        assert flags.cpu().tolist() == [launch] * total + [0]


@pytest.mark.parametrize("M,N,K,BM,BN,parts,aa,ba,name", [
    (100, 200, 1030, 64, 64, 3, False, True, "64x64x128_w2x2_gather"),    # the owner's hand-over, parts of an odd and an even number of steps
    (100, 200, 1030, 64, 64, 8, True, True, "64x64x128_w2x2_gather"),     # sliced
    (256, 136, 1023, 128, 128, 4, False, True, "128x128x64_w2x2_gather"),
    (256, 136, 1023, 128, 128, 4, False, False, "128x128x64_w2x2_s4_f4_gather_dma"),
    (200, 72, 779, 256, 64, 4, False, True, "256x64x64_w4x1_gather"),
    (300, 250, 1025, 256, 128, 2, False, True, "256x128x64_w2x2_gather"),  # a 128-accumulator tile: the pair hand-over
    (30, 250, 1025, 64, 128, 16, True, False, "64x128x64_w2x2_gather"),   # parts of one step
])
def test_split_k(shmem, M, N, K, BM, BN, parts, aa, ba, name):
    dtype, grid = BF16, 64
    A, B = make_ab(M, N, K, dtype)
    a = place(shmem, A, aa, 1, 0)
    b = place(shmem, B, False, 1, 0) if ba else place(shmem, B.T, False, 1, 0).T
    cg = shmem.zeros((M, N), dtype=dtype)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total,), dtype=torch.int32)
    P = shmem.zeros((grid, BM * BN), dtype=F32)
    locks = shmem.zeros((grid,), dtype=torch.int32)
    args = (a, b, None, cg, flags, None, 0, 1, grid, BM, BN, 64, 2, ops.EPI_ALL_SCATTER)
    kw = dict(partials=P, locks=locks, split_k=parts)
    assert ops.gemm_plan_name(*args, **kw) == name
    for launch in (1, 2):
        ops.gemm_launch(*args, **kw)
        torch.cuda.synchronize()
        check_close(cg, O.shard_gemm(A, B, dtype), f"launch {launch}")
        assert flags.cpu().tolist() == [launch] * total and not locks.any()


@pytest.mark.parametrize("phase", [ops.PHASE_FUSED, ops.PHASE_TWO_KERNELS])
@pytest.mark.parametrize("BM,BN", [(64, 64), (128, 128), (256, 64), (64, 128)])
def test_one_shot_of_a_row_major_weight(shmem, BM, BN, phase):
    """world_size 1: the partial is stored, c_global is its cast."""
    M, N, K, dtype = 150, 213, 333, F16
    A, B = make_ab(M, N, K, dtype)
    a, b = place(shmem, A, False, 0, 0), place(shmem, B, False, 0, 0)
    c = shmem.zeros((M, N), dtype=F32)
    cg = shmem.zeros((M, N), dtype=dtype)
    flags = shmem.zeros((ops.cdiv(M, BM) * ops.cdiv(N, BN),), dtype=torch.int32)
    args = (a, b, c, cg, flags, shmem.get_heap_bases(), 0, 1, 8, BM, BN, 64, 6, ops.EPI_ONE_SHOT)
    name = ops.gemm_plan_name(*args, phase=phase)
    assert name.endswith("_gather+reduce" if phase == ops.PHASE_FUSED else "_gather")
    ops.gemm_launch(*args, phase=phase)
    torch.cuda.synchronize()
    check_close(c, O.shard_gemm(A, B, F32), "partial")
    assert torch.equal(cg.cpu(), O.one_shot_reduce(c.cpu()[None], dtype))


@pytest.mark.parametrize("out_dtype", [F32, F16])
def test_atomic_accumulate_of_odd_k_shards(shmem, out_dtype):
    M, N, ks, ws, dtype = 200, 136, 67, 4, F16
    A, B = make_ab(M, N, ks * ws, dtype)
    a, b = place(shmem, A, False, 1, 1), place(shmem, B, False, 0, 0)
    cg = shmem.zeros((M, N), dtype=out_dtype)
    for r in range(ws):
        args = (a[:, r * ks:(r + 1) * ks], b[r * ks:(r + 1) * ks, :], None, cg, None, None, 0, 1, 8, 128, 128, 64, 6, ops.EPI_ATOMIC_ADD)
        assert ops.gemm_plan_name(*args) == "128x128x64_w2x2_gather"
        ops.gemm_launch(*args)
    torch.cuda.synchronize()
    want = O.atomics_all_reduce(O.k_shards(A, B, ws))
    check_close(cg, want, "sum", block_rtol=2 ** -7 if out_dtype == F32 else None)
