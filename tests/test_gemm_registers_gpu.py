"""The 128-accumulator tiles with fetching waves sit at the edge of a wave's 256 registers: their unsplit store builds
keep everything in them, no scratch."""

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
