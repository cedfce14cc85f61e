"""The few-rows kernel and the cells with the one-shot reduce inside: partials and flags as those of the kernel without it, the
result bit for bit the sum of the partials in rank order, whether the peers have signalled before the launch, while it
waits for them, or not at all."""

import pytest
import torch

from iris_amd import ops
from oracle import iris_oracle as O
from parity import check_close, make_ab
from test_concurrent_gpu import two_streams  # noqa: F401  (a fixture)
from test_gemm_gather_gpu import place

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


class Ranks:
    """`ws` ranks' shards of one product, their buffers, and launches of one rank's share."""

    def __init__(self, shmem, M, N, ks, BM, BN, ws, dtype, part, out, rows=False, programs=256):
        self.shmem, self.ws, self.total = shmem, ws, ops.cdiv(M, BM) * ops.cdiv(N, BN)
        A, B = make_ab(M, N, ks * ws, dtype)
        a = place(shmem, A, False, 0, 0)
        b = place(shmem, B, False, 0, 0) if rows else place(shmem, B.T, False, 0, 0).T
        self.shards = O.k_shards(A, B, ws)
        self.part, self.out = shmem.zeros((M, N), dtype=part), shmem.zeros((M, N), dtype=out)
        self.flags = shmem.zeros((self.total,), dtype=torch.int32)
        self.P = [torch.zeros((programs, max(BM * BN, 1024)), dtype=F32, device="cuda") for _ in range(ws)]
        self.locks = [torch.zeros((programs,), dtype=torch.int32, device="cuda") for _ in range(ws)]
        self.status = torch.zeros(1, dtype=torch.int32, device="cuda")
        on = shmem.on_rank
        for r in range(ws):
            on(self.part, r).zero_(), on(self.flags, r).zero_(), on(self.out, r).fill_(-7)
        self.args = [(a[:, r * ks:(r + 1) * ks], b[r * ks:(r + 1) * ks, :], on(self.part, r), on(self.out, r), on(self.flags, r),
                      shmem.get_heap_bases(), r, ws, programs, BM, BN, 64, 3, ops.EPI_ONE_SHOT) for r in range(ws)]

    def launch(self, r, phase, **kw):
        space = dict(partials=self.P[r], locks=self.locks[r], num_xcds=8)
        ops.gemm_launch(*self.args[r], phase=phase, status=self.status, **space, **kw)
        return ops.gemm_plan_name(*self.args[r], phase=phase, **space)

    def check(self, r):
        on = self.shmem.on_rank
        parts = torch.stack([on(self.part, q).cpu() for q in range(self.ws)])
        for q in range(self.ws):
            check_close(parts[q], O.shard_gemm(*self.shards[q], self.part.dtype), f"partial {q}")
        assert torch.equal(on(self.out, r).cpu(), O.one_shot_reduce(parts, self.out.dtype))
        assert not on(self.flags, r).any() and int(self.status.item()) == 0
        assert not any(x.any() for x in self.locks)


@pytest.mark.parametrize("M,N,ks,BM,BN,ws,dtype,part,out,rows,kernel", [
    (1, 64, 64, 64, 64, 2, BF16, BF16, BF16, False, "few_rows_16xN"),       # one tile, one block of K
    (16, 4096, 1376, 64, 64, 8, BF16, F32, BF16, False, "few_rows_16xN"),
    (9, 203, 192, 64, 64, 4, BF16, BF16, BF16, False, "few_rows_16xN"),     # rows of an odd length, N inside a lane's columns
    (7, 130, 320, 64, 64, 3, F16, F16, F32, False, "few_rows_16xN"),
    (17, 272, 256, 64, 128, 4, F16, F32, F16, False, "few_rows_16xN"),      # two blocks of rows a tile
    (5, 77, 512, 64, 64, 8, F32, F32, F32, False, "few_rows_16xN"),
    (3, 192, 8192, 64, 64, 4, BF16, BF16, BF16, False, "few_rows_16xN"),    # K shared out over workgroups
    (50, 300, 2112, 64, 64, 2, BF16, F32, BF16, False, "few_rows_32xN"),
    (9, 201, 1031, 64, 64, 4, BF16, F32, BF16, False, "few_rows_16xN_gather_dma"),
    (100, 131, 640, 64, 64, 2, BF16, BF16, BF16, False, "cells_32x32"),
    (100, 264, 640, 128, 64, 4, F16, F16, F16, False, "cells_32x32"),
    (100, 264, 520, 64, 64, 4, BF16, F32, BF16, True, "cells_32x32_rows"),
    (13, 328, 520, 64, 64, 8, BF16, BF16, BF16, True, "cells_16x32_rows"),
])
@pytest.mark.parametrize("kw", [{}, dict(scope=ops.SCOPE_SYSTEM, flag_sem=ops.FLAG_SEM_RELEASE_ACQUIRE)])
def test_peers_are_done(shmem, M, N, ks, BM, BN, ws, dtype, part, out, rows, kernel, kw):
    job = Ranks(shmem, M, N, ks, BM, BN, ws, dtype, part, out, rows)
    last = ws // 2
    for r in range(ws):
        if r != last:
            job.launch(r, ops.PHASE_PRODUCE, **kw)
    assert job.launch(last, ops.PHASE_TWO_KERNELS, **kw) == kernel
    torch.cuda.synchronize()
    job.check(last)
    for r in range(ws):
        if r != last:
            assert shmem.on_rank(job.flags, r).cpu().tolist() == [ws - 1] * job.total
    # a second round on the same buffers
    shmem.on_rank(job.flags, last).fill_(ws - 1)
    job.launch(last, ops.PHASE_FUSED, **kw)
    torch.cuda.synchronize()
    job.check(last)


@pytest.mark.parametrize("M,N,ks,part,rows", [(16, 1024, 1376, F32, False), (9, 203, 192, BF16, False), (3, 192, 8192, BF16, False),
                                              (60, 200, 520, BF16, True)])
@pytest.mark.parametrize("kw", [{}, dict(scope=ops.SCOPE_SYSTEM, flag_sem=ops.FLAG_SEM_RELEASE_ACQUIRE)])
def test_peers_come_later(shmem, two_streams, M, N, ks, part, rows, kw):  # noqa: F811
    """The reducing launch is enqueued first and its last workgroup of a tile waits for the peer, which comes on another
    stream."""
    job = Ranks(shmem, M, N, ks, 64, 64, 2, BF16, part, BF16, rows)
    waits, comes = two_streams
    on = shmem.on_rank
    job.launch(1, ops.PHASE_PRODUCE, **kw)  # (loaded, and the partials in place)
    torch.cuda.synchronize()
    for _ in range(20):
        on(job.flags, 0).zero_(), on(job.flags, 1).zero_(), on(job.out, 0).fill_(-7)
        torch.cuda.synchronize()
        with torch.cuda.stream(waits):
            job.launch(0, ops.PHASE_TWO_KERNELS, spin_timeout_ticks=50_000_000, **kw)
        with torch.cuda.stream(comes):
            job.launch(1, ops.PHASE_PRODUCE, **kw)
        torch.cuda.synchronize()
        job.check(0)


def test_a_peer_that_does_not_come(shmem):
    """Tiles whose flag does not arrive keep their count and their part of the result; the others are reduced."""
    M, N, ws = 12, 200, 3
    job = Ranks(shmem, M, N, 256, 64, 64, ws, BF16, F32, BF16)
    on = shmem.on_rank
    for r in (0, 1):
        job.launch(r, ops.PHASE_PRODUCE)
    torch.cuda.synchronize()
    on(job.flags, 2)[1:3] = 1
    job.launch(2, ops.PHASE_TWO_KERNELS, spin_timeout_ticks=2000)
    torch.cuda.synchronize()
    assert int(job.status.item()) == 1 and on(job.flags, 2).cpu().tolist() == [0, 1, 1, 0]
    assert not any(x.any() for x in job.locks)
    parts = torch.stack([on(job.part, q).cpu() for q in range(ws)])
    want = O.one_shot_reduce(parts, BF16)
    want[:, 64:192] = -7
    assert torch.equal(on(job.out, 2).cpu(), want)
    job.status.zero_()
    on(job.flags, 2)[1:3] = 2
    on(job.flags, 2)[0], on(job.flags, 2)[3] = 2, 2
    job.launch(2, ops.PHASE_TWO_KERNELS)
    torch.cuda.synchronize()
    job.check(2)
