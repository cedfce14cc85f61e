"""Launches whose tiles are parts of the caller's: every flag is raised once
per launch, by the part that counts last, on every rank; the counters are left
at zero; values against the CPU oracle.  One-part tiles at ragged edges, split
parts, all operand kinds, and where the launcher keeps the caller's tiles."""

import pytest
import torch

from iris_amd import ops
from oracle import iris_oracle as O
from parity import check_close, make_ab
from test_gemm_gather_gpu import place

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("M,N,K,BM,BN,grid,ws,dtype,odd,plan,split", [
    (300, 200, 192, 256, 256, 256, 2, BF16, False, "64x64x128_w2x2_s4_f4", 1),     # 2 x 1 tiles in 5 x 4 parts
    (300, 200, 192, 256, 256, 248, 1, BF16, False, None, 1),                       # not the whole device
    (1100, 1000, 200, 256, 128, 256, 1, F16, False, "128x64x64_w2x2_s4_f4", 1),    # 64 x 64: 288 parts
    (100, 16000, 200, 64, 256, 256, 1, BF16, False, "64x128x64_w2x2_s4_f4", 1),    # tiles 64 rows high
    (1600, 2100, 136, 256, 256, 256, 1, BF16, False, "128x128x64_w2x2_s4_f4", 1),  # 128 x 64: 429 parts
    (2100, 2100, 136, 256, 256, 256, 1, BF16, False, None, 1),                     # too many parts for the programs
    (200, 140, 2048, 128, 128, 256, 3, BF16, False, "64x64x128_w2x2_s4_f4", 8),    # parts of parts
    (200, 140, 4096, 128, 64, 256, 1, F16, False, "64x64x128_w2x2_s4_f4", 16),
    (300, 201, 301, 256, 64, 256, 2, F16, True, "64x64x128_w2x2_gather", 1),
    (500, 601, 2051, 128, 128, 256, 1, BF16, True, "64x64x128_w2x2_gather", 2),    # (three, but for the flags' words)
    (300, 200, 516, 256, 128, 256, 2, F32, False, "64x64x64_w2x2_s4_f4_fp32", 4),
])
def test_scatter(shmem, M, N, K, BM, BN, grid, ws, dtype, odd, plan, split):
    A, B = make_ab(M, N, K, dtype)
    a = place(shmem, A, False, 0, 0)
    b = place(shmem, B, False, 0, 0) if odd else place(shmem, B.T, False, 0, 0).T
    cg = shmem.zeros((M, N * ws), dtype=dtype)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total + 2,), dtype=torch.int32)
    for r in range(ws):
        shmem.on_rank(cg, r).zero_()
        shmem.on_rank(flags, r).zero_()
    P = shmem.zeros((grid, BM * BN), dtype=F32)
    locks = shmem.zeros((grid,), dtype=torch.int32)
    args = (a, b, None, cg, flags, shmem.get_heap_bases(), 0, ws, grid, BM, BN, 64, 2, ops.EPI_ALL_SCATTER)
    # (a small product of a launch that knows its XCDs runs in cells of 32 x 32 instead)
    kw = dict(partials=P, locks=locks, num_xcds=1 if M * N <= 1 << 18 else ops.default_num_xcds(256, grid))
    name = ops.gemm_plan_name(*args, **kw)
    assert name == plan + "+parts_of_tiles" if plan else "parts" not in name
    assert ops.gemm_split_k(*args, **kw) == split
    want = O.shard_gemm(A, B, dtype)
    for launch in (1, 2, 3):
        ops.gemm_launch(*args, **kw)
        torch.cuda.synchronize()
        for r in range(ws):
            check_close(shmem.on_rank(cg, r)[:, :N], want, f"launch {launch}, rank {r}")
            assert shmem.on_rank(flags, r).cpu().tolist() == [launch] * total + [0, 0]
        assert not locks.any()
    # without the counters' words the caller's tiles stay
    assert "parts" not in ops.gemm_plan_name(*args, num_xcds=kw["num_xcds"])
    if split == 1:  # ... and the no-allocation launch has words of its own
        ops.gemm_launch(*args, num_xcds=kw["num_xcds"], noalloc=True)
        torch.cuda.synchronize()
        check_close(cg[:, :N], want, "no allocation")
        assert flags.cpu().tolist() == [4] * total + [0, 0]


def test_one_shot_and_atomics(shmem):
    """The producer's signal (other ranks' flags only), and an epilogue without flags, which needs no counters."""
    ws, M, N, ks, BM, BN = 4, 300, 264, 192, 256, 128
    A, B = make_ab(M, N, ks * ws, BF16)
    a, b = place(shmem, A, False, 0, 0), place(shmem, B.T, False, 0, 0).T
    shards = O.k_shards(A, B, ws)
    c, cg = shmem.zeros((M, N), dtype=F32), shmem.zeros((M, N), dtype=BF16)
    total = ops.cdiv(M, BM) * ops.cdiv(N, BN)
    flags = shmem.zeros((total,), dtype=torch.int32)
    acc = shmem.zeros((M, N), dtype=F32)
    P, locks = shmem.zeros((256, BM * BN), dtype=F32), shmem.zeros((256,), dtype=torch.int32)
    for r in range(ws):
        for t in (c, cg, flags):
            shmem.on_rank(t, r).zero_()
    for r in range(ws):
        args = (a[:, r * ks:(r + 1) * ks], b[r * ks:(r + 1) * ks, :], shmem.on_rank(c, r), shmem.on_rank(cg, r),
                shmem.on_rank(flags, r), shmem.get_heap_bases(), r, ws, 256, BM, BN, 64, 6, ops.EPI_ONE_SHOT)
        kw = dict(phase=ops.PHASE_FUSED if r == ws - 1 else ops.PHASE_PRODUCE, partials=P, locks=locks)
        assert "+parts_of_tiles" in ops.gemm_plan_name(*args, **kw)
        ops.gemm_launch(*args, **kw)
        ops.gemm_launch(args[0], args[1], None, acc, None, None, 0, 1, 256, BM, BN, 64, 6, ops.EPI_ATOMIC_ADD)
    torch.cuda.synchronize()
    for r in range(ws):
        check_close(shmem.on_rank(c, r), O.shard_gemm(*shards[r], F32), f"partial {r}")
        assert shmem.on_rank(flags, r).cpu().tolist() == [0 if r == ws - 1 else ws - 1] * total
    check_close(shmem.on_rank(cg, ws - 1), O.one_shot_all_reduce(shards, F32, BF16), "reduced")
    check_close(acc, O.atomics_all_reduce(shards), "atomics")
    assert not locks.any()
