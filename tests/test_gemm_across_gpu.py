"""Launches whose tiles lie across the caller's: parts of them, blocks, and tiles that share two or more of the caller's each; K
whole and in parts with each hand-over.  Every flag is raised once per launch on every rank, the counters are left at zero (in
words and in bytes of words), values against the CPU oracle."""

import pytest
import torch

from iris_amd import ops
from oracle import iris_oracle as O
from parity import check_close, make_ab
from test_gemm_gather_gpu import place

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("M,N,K,BM,BN,dtype,out,rows,kernel,parts", [
    (1911, 2120, 472, 256, 64, BF16, BF16, False, "128x128x64_w2x2_s4_f4", 1),     # two columns of the caller's, half of their rows
    (1219, 1016, 1168, 64, 64, BF16, BF16, False, "128x64x64_w2x2_s4_f4", 1),      # blocks of the caller's; 320 tiles, in bytes
    (1803, 2688, 288, 256, 256, F16, F16, False, "256x128x64_w2x2_s3_f4", 1),      # halves
    (2497, 1544, 2272, 128, 128, BF16, BF16, False, "256x64x64_w4x1_s3_f4", 1),
    (838, 1088, 1536, 256, 256, BF16, BF16, False, "64x64x128_w2x2_s4_f4", 1),
    (2085, 984, 2168, 64, 64, BF16, F32, False, "128x128x64_w2x2_s4_f4", 1),
    (1903, 200, 8624, 256, 64, BF16, BF16, False, "128x128x64_w2x2_s4_f4", 8),     # sliced
    (1303, 328, 7912, 256, 64, BF16, F32, False, "128x128x64_w2x2_s4_f4", 7),      # the owner's
    (172, 2456, 6480, 128, 128, F16, F16, False, "64x128x64_w2x2_s4_f4", 4),
    (421, 1728, 10696, 256, 256, BF16, BF16, False, "256x128x64_w2x2_s3_f4", 9),
    (241, 1272, 6328, 256, 64, BF16, BF16, False, "64x64x128_w2x2_s4_f4", 3),
    (856, 1296, 304, 64, 64, F32, F32, False, "64x128x32_w2x2_s4_f4_fp32", 1),
    (225, 2408, 1608, 256, 64, F32, F32, False, "64x128x32_w2x2_s4_f4_fp32", 3),
    (917, 1160, 240, 64, 64, BF16, BF16, True, "64x128x64_w2x2_s4_f4_rows", 1),
    (333, 1320, 6144, 256, 64, BF16, BF16, True, "128x128x64_w2x2_s4_f4_rows", 7),
    (1285, 2115, 202, 64, 64, BF16, BF16, False, "128x128x64_w2x2_s4_f4_gather_dma", 1),
    (135, 2511, 7522, 256, 64, BF16, BF16, False, "64x128x64_w2x2_s4_f4_gather_dma", 4),
])
def test_scatter(shmem, M, N, K, BM, BN, dtype, out, rows, kernel, parts):
    ws = 2
    A, B = make_ab(M, N, K, dtype)
    a = place(shmem, A, False, 0, 0)
    b = place(shmem, B, False, 0, 0) if rows else place(shmem, B.T, False, 0, 0).T
    cg = shmem.zeros((M, N * ws), dtype=out)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total + 2,), dtype=torch.int32)
    P, locks = shmem.zeros((256, BM * BN), dtype=F32), shmem.zeros((256,), dtype=torch.int32)
    for r in range(ws):
        shmem.on_rank(cg, r).zero_(), shmem.on_rank(flags, r).zero_()
    args = (a, b, None, cg, flags, shmem.get_heap_bases(), 0, ws, 256, BM, BN, 64, 4, ops.EPI_ALL_SCATTER)
    kw = dict(partials=P, locks=locks, num_xcds=8)
    assert (ops.gemm_plan_name(*args, **kw), ops.gemm_split_k(*args, **kw)) == (kernel + "+across_the_tiles", parts)
    want = O.shard_gemm(A, B, out)
    for launch in (1, 2, 3):
        ops.gemm_launch(*args, **kw)
        torch.cuda.synchronize()
        for r in range(ws):
            check_close(shmem.on_rank(cg, r)[:, :N], want, f"launch {launch}, rank {r}")
            assert shmem.on_rank(flags, r).cpu().tolist() == [launch] * total + [0, 0]
        assert not locks.any()
    # flags that are releases, and a launch without the counters, keep the caller's tiles
    assert "across" not in ops.gemm_plan_name(*args, num_xcds=8)
    ops.gemm_launch(*args, flag_sem=ops.FLAG_SEM_RELEASE_ACQUIRE, **kw)
    torch.cuda.synchronize()
    assert flags.cpu().tolist() == [4] * total + [0, 0] and not locks.any()


@pytest.mark.parametrize("M,N,ks,BM,BN,dtype", [(1911, 2120, 512, 256, 64, BF16), (1805, 2688, 320, 256, 256, BF16), (856, 1296, 304, 64, 64, F32)])
def test_one_shot(shmem, M, N, ks, BM, BN, dtype):
    """The producer's signal, and the reduce behind it."""
    ws = 2
    A, B = make_ab(M, N, ks * ws, dtype)
    a, b = place(shmem, A, False, 0, 0), place(shmem, B.T, False, 0, 0).T
    shards = O.k_shards(A, B, ws)
    c, cg = shmem.zeros((M, N), dtype=dtype), shmem.zeros((M, N), dtype=dtype)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total,), dtype=torch.int32)
    P, locks = shmem.zeros((256, BM * BN), dtype=F32), shmem.zeros((256,), dtype=torch.int32)
    for r in range(ws):
        for t in (c, cg, flags):
            shmem.on_rank(t, r).zero_()
    for r in range(ws):
        args = (a[:, r * ks:(r + 1) * ks], b[r * ks:(r + 1) * ks, :], shmem.on_rank(c, r), shmem.on_rank(cg, r), shmem.on_rank(flags, r),
                shmem.get_heap_bases(), r, ws, 256, BM, BN, 64, 4, ops.EPI_ONE_SHOT)
        kw = dict(phase=ops.PHASE_TWO_KERNELS if r == 1 else ops.PHASE_PRODUCE, partials=P, locks=locks, num_xcds=8)
        assert "+across_the_tiles" in ops.gemm_plan_name(*args, **kw)
        ops.gemm_launch(*args, **kw)
    torch.cuda.synchronize()
    got = torch.stack([shmem.on_rank(c, r).cpu() for r in range(ws)])
    for r in range(ws):
        check_close(got[r], O.shard_gemm(*shards[r], dtype), f"partial {r}")
        assert shmem.on_rank(flags, r).cpu().tolist() == [0 if r == 1 else 1] * total
    assert torch.equal(shmem.on_rank(cg, 1).cpu(), O.one_shot_reduce(got, dtype)) and not locks.any()
