"""The 128-accumulator tiles with fetching waves sit at the edge of a wave's 256 registers: their unsplit store builds
for operands along K keep everything in them, no scratch; those for a row-major B (``_rows``) and for operands at any alignment
(``_gather_dma``) spill up to 24 bytes a lane, none of it in a K-step, in the 256 x 128 tile, and nothing in the others."""

import pytest
import torch

from iris_amd import ops

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("M,N,K,BM,BN,variant,name", [
    (2048, 4096, 1024, 256, 128, 0, "256x128x64_w2x2_s3_f4"),
    (4096, 2048, 1024, 128, 256, 0, "128x256x64_w1x4_s3_f4"),
    (8192, 1024, 1024, 256, 64, 0, "256x128x64_w2x2_s3_f4+two_tiles_each"),
])
@pytest.mark.parametrize("dtype,out", [(BF16, BF16), (F16, F16), (BF16, F32), (F16, F32)])
def test_no_scratch(shmem, M, N, K, BM, BN, variant, name, dtype, out):
    a, b = torch.empty((M, K), dtype=dtype, device="cuda"), torch.empty((N, K), dtype=dtype, device="cuda").T
    cg = shmem.zeros((M, N), dtype=out)
    flags = shmem.zeros((ops.cdiv(M, BM) * ops.cdiv(N, BN),), dtype=torch.int32)
    args = (a, b, None, cg, flags, shmem.get_heap_bases(), 0, 1, 256, BM, BN, 64, 4, ops.EPI_ALL_SCATTER)
    assert ops.gemm_plan_name(*args, variant=variant, num_xcds=8) == name
    registers, scratch = ops.gemm_kernel_info(*args, variant=variant, num_xcds=8)
    assert registers <= 256 and scratch == 0


@pytest.mark.parametrize("M,N,K,BM,BN,variant,name,most", [
    (2048, 4096, 1024, 256, 256, 0, "256x256x64_w2x4_s2%s", ((0, 0), (0, 0))),
    (8192, 1344, 4096, 256, 128, 0, "256x256x64_w2x4_s2%s+two_tiles_each", ((0, 0), (0, 0))),
    (2048, 4096, 1024, 256, 128, 0, "256x128x64_w2x2_s3_f4%s", ((20, 0), (24, 8))),
    (8192, 1024, 1024, 256, 64, 0, "256x128x64_w2x2_s3_f4%s+two_tiles_each", ((12, 0), (16, 0))),
    (2048, 1024, 1024, 128, 128, ops.VARIANT_PERSISTENT, "128x128x64_w2x2_s4_f4%s", ((0, 0), (0, 0))),
    (2048, 1024, 1024, 256, 64, ops.VARIANT_PERSISTENT, "256x64x64_w4x1_s3_f4%s", ((0, 0), (0, 0))),
    (2048, 1024, 1024, 128, 64, ops.VARIANT_PERSISTENT, "128x64x64_w2x2_s4_f4%s", ((0, 0), (0, 0))),
    (2048, 1024, 1024, 64, 128, ops.VARIANT_PERSISTENT, "64x128x64_w2x2_s4_f4%s", ((0, 0), (0, 0))),
    (1024, 1024, 1024, 64, 64, ops.VARIANT_PERSISTENT, "64x64x128_w2x2_s4_f4%s", ((0, 0), (0, 0))),
])
@pytest.mark.parametrize("kind", ["_rows", "_gather_dma"])
@pytest.mark.parametrize("dtype,out", [(BF16, BF16), (F16, F16), (BF16, F32), (F16, F32)])
def test_scratch_of_other_operands(shmem, M, N, K, BM, BN, variant, name, most, kind, dtype, out):
    rows = kind == "_rows"
    K += not rows
    a = torch.empty((M, K), dtype=dtype, device="cuda")
    b = torch.empty((K, N) if rows else (N, K), dtype=dtype, device="cuda")
    cg = shmem.zeros((M, N), dtype=out)
    flags = shmem.zeros((ops.cdiv(M, BM) * ops.cdiv(N, BN),), dtype=torch.int32)
    args = (a, b if rows else b.T, None, cg, flags, shmem.get_heap_bases(), 0, 1, 256, BM, BN, 64, 4, ops.EPI_ALL_SCATTER)
    assert ops.gemm_plan_name(*args, variant=variant, num_xcds=8) == name % kind
    registers, scratch = ops.gemm_kernel_info(*args, variant=variant, num_xcds=8)
    assert registers <= 256 and scratch <= most[kind == "_gather_dma"][out == F32]
