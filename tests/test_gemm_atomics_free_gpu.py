"""Atomic launches in other tiles than the caller's, and with K shared out over programs that each add their own sums: added
to what C holds on every rank, at the edges of tiles and of parts, with and without the callers' workspace."""

import pytest
import torch

from iris_amd import ops
from oracle import iris_oracle as O
from parity import check_close, make_ab
from test_gemm_gather_gpu import place

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("M,N,K,BM,BN,dtype,out,rows,ws,kernel,parts", [
    # K in parts that each add their sums: even and uneven parts, rows and columns past the edges
    (1393, 1520, 3928, 64, 64, F16, F32, False, 1, "128x256x64_w1x4_s3_f4", 3),
    (1318, 1581, 3821, 256, 64, F16, F32, False, 1, "256x128x64_w2x2_s3_f4_gather_dma", 3),
    (266, 1152, 6248, 64, 64, BF16, F32, False, 1, "64x128x64_w2x2_s4_f4", 5),
    (924, 1128, 3224, 256, 64, BF16, F32, False, 1, "128x128x64_w2x2_s4_f4", 3),
    (965, 1296, 4504, 128, 128, BF16, F32, False, 1, "256x64x64_w4x1_s3_f4", 3),
    (1158, 283, 4087, 64, 64, BF16, F32, False, 1, "128x64x64_w2x2_s4_f4_gather_dma", 5),
    (450, 2080, 3176, 64, 64, BF16, F32, True, 1, "128x128x64_w2x2_s4_f4_rows", 3),
    (1145, 320, 272, 256, 64, F32, F32, False, 2, "64x128x32_w2x2_s4_f4_fp32", 3),
    (531, 1824, 664, 256, 64, F32, F32, False, 1, "128x128x32_w2x2_s4_f4_fp32", 3),
    # another tile
    (883, 1408, 280, 256, 64, F32, F32, False, 1, "64x128x32_w2x2_s4_f4_fp32", 1),
    (461, 2104, 1176, 64, 64, BF16, F32, False, 1, "128x64x64_w2x2_s4_f4", 1),
    (1253, 2464, 1008, 64, 64, BF16, BF16, False, 1, "128x128x64_w2x2_s4_f4", 1),   # whole sums, rounded once
])
@pytest.mark.parametrize("workspace", [True, False])
def test_added_to_c(shmem, M, N, K, BM, BN, dtype, out, rows, ws, kernel, parts, workspace):
    A, B = make_ab(M, N, K, dtype)
    a = place(shmem, A, False, 0, 0)
    b = place(shmem, B, False, 0, 0) if rows else place(shmem, B.T, False, 0, 0).T
    c = shmem.zeros((M, N), dtype=out)
    space = {}
    if workspace:
        space = dict(partials=torch.zeros((256, BM * BN), device="cuda"), locks=torch.zeros((256,), dtype=torch.int32, device="cuda"))
    for r in range(ws):
        shmem.on_rank(c, r).fill_(r + 1)
    args = (a, b, None, c, None, shmem.get_heap_bases(), 0, ws, 256, BM, BN, 64, 4, ops.EPI_ATOMIC_ADD)
    plan = ops.gemm_plan_name(*args, num_xcds=8, **space), ops.gemm_split_k(*args, num_xcds=8, **space)
    assert plan == (kernel, parts) or not workspace
    for _ in range(2):
        ops.gemm_launch(*args, num_xcds=8, **space)
    torch.cuda.synchronize()
    want = O.shard_gemm(A, B, F32)
    for r in range(ws):
        got = shmem.on_rank(c, r).float().cpu()
        if out == F32:
            check_close((got - (r + 1)) / 2, want, f"rank {r}")
        else:  # (two sums rounded as they come in, beside a one)
            check_close(got, 2 * want + r + 1, f"rank {r}")
    if workspace:
        assert not space["locks"].any()


def test_what_is_asked_for_is_kept(shmem):
    """A number of parts, a tile by number, timestamps, fewer programs than CUs."""
    A, B = make_ab(965, 1296, 4504, F16)
    a, b = place(shmem, A, False, 0, 0), place(shmem, B.T, False, 0, 0).T
    c = shmem.zeros((965, 1296), dtype=F32)
    P, locks = torch.zeros((256, 128 * 128), device="cuda"), torch.zeros((256,), dtype=torch.int32, device="cuda")

    def name(programs=256, **kw):
        return ops.gemm_plan_name(a, b, None, c, None, shmem.get_heap_bases(), 0, 1, programs, 128, 128, 64, 4, ops.EPI_ATOMIC_ADD,
                                  num_xcds=8, partials=P, locks=locks, **kw)
    assert name().startswith("256x64x64")
    assert name(split_k=1).startswith("128x128") and name(split_k=2).startswith("128x128")
    assert name(variant=4).startswith("128x128") and name(programs=248).startswith("128x128")
