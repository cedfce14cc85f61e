"""fp32 operands with a K of eight K-steps or more: the tiles behind the fp32
table (the scripts' 256 x 64 as one compute tile, split K, the gathering
loader) against the CPU oracle, every 16 x 16 block within 1e-4 of its norm."""

import pytest
import torch

from iris_amd import ops
from oracle import iris_oracle as O
from parity import check_close, make_ab
from test_gemm_gather_gpu import place

pytestmark = pytest.mark.gpu

F32 = torch.float32


@pytest.mark.parametrize("M,N,K,BM,BN,grid,ws,row_major,plan,parts", [
    (520, 200, 256, 256, 64, 4, 1, False, "256x64x32_w4x1_s3_f4_fp32", 1),     # eight K-steps, three tiles a program
    (520, 200, 252, 256, 64, 4, 1, False, "64x64x32_w2x2_s4_fp32", 1),         # one element short of them
    (300, 250, 1028, 256, 64, 256, 2, False, "256x64x32_w4x1_s3_f4_fp32", 8),  # sliced
    (300, 250, 1028, 128, 128, 32, 1, False, "128x128x32_w2x2_s4_f4_fp32", 5),  # the owner's hand-over
    (24, 200, 2052, 256, 64, 256, 1, False, "64x64x64_w2x2_s4_f4_fp32", 16),
    (40, 260, 1024, 64, 128, 16, 1, False, "64x128x32_w2x2_s4_f4_fp32", 5),
    (300, 200, 1030, 256, 64, 64, 1, True, "256x64x32_w4x1_gather_fp32", 8),
    (257, 129, 515, 128, 128, 8, 1, True, "128x128x32_w2x2_gather_fp32", 1),   # an odd K, row-major B
    (100, 75, 1025, 64, 64, 64, 1, False, "64x64x64_w2x2_gather_fp32", 8),     # an odd K along the rows
])
def test_scatter(shmem, M, N, K, BM, BN, grid, ws, row_major, plan, parts):
    A, B = make_ab(M, N, K, F32)
    a = place(shmem, A, False, 0, 0)
    b = place(shmem, B, False, 0, 0) if row_major else place(shmem, B.T, False, 0, 0).T
    cg = shmem.zeros((M, N * ws), dtype=F32)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total,), dtype=torch.int32)
    for r in range(ws):
        shmem.on_rank(cg, r).zero_()
        shmem.on_rank(flags, r).zero_()
    P = shmem.zeros((grid, BM * BN), dtype=F32)
    locks = shmem.zeros((grid,), dtype=torch.int32)
    args = (a, b, None, cg, flags, shmem.get_heap_bases(), 0, ws, grid, BM, BN, 64, 2, ops.EPI_ALL_SCATTER)
    kw = dict(partials=P, locks=locks, split_k=parts if parts > 1 else 0)
    assert ops.gemm_plan_name(*args, **kw) == plan and ops.gemm_split_k(*args, **kw) == parts
    want = O.shard_gemm(A, B, F32)
    for launch in (1, 2):
        ops.gemm_launch(*args, **kw)
        torch.cuda.synchronize()
        for r in range(ws):
            check_close(shmem.on_rank(cg, r)[:, :N], want, f"launch {launch}, rank {r}", block_rtol=1e-4)
            assert shmem.on_rank(flags, r).cpu().tolist() == [launch] * total
        assert not locks.any()


def test_atomic_accumulate_of_k_shards(shmem):
    M, N, ks, ws = 300, 136, 260, 3
    A, B = make_ab(M, N, ks * ws, F32)
    a, b = place(shmem, A, False, 0, 0), place(shmem, B.T, False, 0, 0).T
    cg = shmem.zeros((M, N), dtype=F32)
    for r in range(ws):
        ops.gemm_launch(a[:, r * ks:(r + 1) * ks], b[r * ks:(r + 1) * ks, :], None, cg, None, None, 0, 1, 8, 256, 64, 64, 6,
                        ops.EPI_ATOMIC_ADD)
    torch.cuda.synchronize()
    check_close(cg, O.atomics_all_reduce(O.k_shards(A, B, ws)), "sum", block_rtol=1e-4)
