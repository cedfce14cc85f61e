"""Launches that reduce as they store, with more late tiles than workgroups may wait: those that wait take the tiles of the
others.  Peers that come while they wait, that do not come, and that share the device with two others that wait."""

import itertools

import pytest
import torch

from iris_amd import ops
from oracle import iris_oracle as O
from parity import check_close
from test_few_rows_reduce_gpu import BF16, F32, Ranks
from test_late_tiles_cpu import kernels

pytestmark = pytest.mark.gpu

HALF_SECOND = 50_000_000  # ticks of the 100 MHz wall clock


@pytest.fixture(scope="module")
def streams(shmem_gpu):
    """Three streams that really run side by side (streams that share a hardware queue do not): each pair of them is probed with
    a one-tile consumer, whose wait is bounded, on one and its signal on the other."""
    shmem = shmem_gpu
    shmem.heap_offset = 0
    c, cg = shmem.zeros((64, 64), dtype=F32), shmem.zeros((64, 64), dtype=F32)
    flags, hb = shmem.zeros((1,), dtype=torch.int32), shmem.get_heap_bases()
    status = torch.zeros(1, dtype=torch.int32, device="cuda")
    made = [torch.cuda.Stream() for _ in range(4)]
    for s in made:  # the first submission to a new stream takes milliseconds
        with torch.cuda.stream(s):
            torch.zeros(8, device="cuda").add_(1)
    torch.cuda.synchronize()

    def apart(sa, sb):
        for r in range(2):
            shmem.on_rank(flags, r).zero_()
        status.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(sb):
            ops.one_shot_reduce(c, cg, flags, hb, 0, 2, 64, 64, 1, num_sms=1, variant=8, status=status, spin_timeout_ticks=2_000_000)
        with torch.cuda.stream(sa):
            ops.signal_tiles(shmem.on_rank(flags, 1), hb, 1, 1, 2)
        torch.cuda.synchronize()
        return int(status.item()) == 0

    ok = {frozenset(p) for p in itertools.combinations(made, 2) if apart(*p) and apart(*reversed(p))}
    for three in itertools.combinations(made, 3):
        if all(frozenset(p) in ok for p in itertools.combinations(three, 2)):
            return three
    pytest.fail("no three streams of this process run side by side on the device")


# (ranks, M, N, K, row-major weight): 64 tiles of four workgroups, 128 of two cells, 21 of K in parts; some of them more than may wait
MANY = [(8, 16, 4096, 1376, False), (8, 16, 8192, 512, True), (8, 3, 1344, 8192, False), (5, 100, 1000, 640, False)]


@pytest.mark.parametrize("ws,M,N,ks,rows", MANY)
@pytest.mark.parametrize("kw", [{}, dict(scope=ops.SCOPE_SYSTEM, flag_sem=ops.FLAG_SEM_RELEASE_ACQUIRE)])
def test_peers_come_later(shmem, streams, ws, M, N, ks, rows, kw):
    layout = dict(stride_bk=N, stride_bn=1) if rows else {}
    n, waiting = kernels(M, N, ks, 64, 64, ws, **layout)
    assert n == 1 and 0 < waiting <= 32 * (7 // (ws - 1))
    job = Ranks(shmem, M, N, ks, 64, 64, ws, BF16, BF16, BF16, rows)
    on, (waits, comes, _) = shmem.on_rank, streams
    for r in range(1, ws):
        job.launch(r, ops.PHASE_PRODUCE, **kw)  # (loaded, and the partials in place)
    torch.cuda.synchronize()
    for _ in range(10):
        for r in range(ws):
            on(job.flags, r).zero_()
        on(job.out, 0).fill_(-7)
        torch.cuda.synchronize()
        with torch.cuda.stream(waits):
            job.launch(0, ops.PHASE_TWO_KERNELS, spin_timeout_ticks=HALF_SECOND, **kw)
        with torch.cuda.stream(comes):
            for r in range(1, ws):
                job.launch(r, ops.PHASE_PRODUCE, **kw)
        torch.cuda.synchronize()
        job.check(0)


@pytest.mark.parametrize("ws,M,N,ks,rows", MANY)
def test_peers_that_do_not_come(shmem, ws, M, N, ks, rows):
    """Every wait ends, tiles that were signalled are reduced whoever they were left to, the others keep their flags."""
    job = Ranks(shmem, M, N, ks, 64, 64, ws, BF16, F32, BF16, rows)
    on = shmem.on_rank
    for r in range(1, ws):
        job.launch(r, ops.PHASE_PRODUCE)
    torch.cuda.synchronize()
    late = torch.arange(job.total, device="cuda") % 3 != 1
    for _ in range(3):
        job.status.zero_()
        on(job.out, 0).fill_(-7)
        on(job.flags, 0).copy_(torch.where(late, ws - 2, ws - 1))
        job.launch(0, ops.PHASE_TWO_KERNELS, spin_timeout_ticks=2000)
        torch.cuda.synchronize()
        assert int(job.status.item()) == 1
        assert torch.equal(on(job.flags, 0), torch.where(late, ws - 2, 0).to(torch.int32))
        assert not any(x.any() for x in job.locks)
    # ... and the words are as they were: the next launch is whole
    job.status.zero_()
    on(job.flags, 0).fill_(ws - 1)
    job.launch(0, ops.PHASE_TWO_KERNELS)
    torch.cuda.synchronize()
    job.check(0)


@pytest.mark.parametrize("M,N,ks,rows", [(16, 8192, 1024, True), (128, 2048, 512, False), (16, 4096, 1376, False)])
def test_three_ranks_side_by_side(shmem, streams, M, N, ks, rows):
    """Each rank's launch signals, waits and reduces; two that wait leave the third room, on every shader engine."""
    ws = 3
    job = Ranks(shmem, M, N, ks, 64, 64, ws, BF16, BF16, BF16, rows)
    on = shmem.on_rank
    torch.cuda.synchronize()
    for _ in range(10):
        for r in range(ws):
            on(job.flags, r).zero_(), on(job.out, r).fill_(-7)
        torch.cuda.synchronize()
        for r, s in enumerate(streams):
            with torch.cuda.stream(s):
                job.launch(r, ops.PHASE_TWO_KERNELS, spin_timeout_ticks=HALF_SECOND)
        torch.cuda.synchronize()
        for r in range(ws):
            job.check(r)


@pytest.mark.parametrize("phase", [ops.PHASE_TWO_KERNELS, ops.PHASE_FUSED])
@pytest.mark.parametrize("over", ["activations", "weights", "partials"])
def test_a_result_in_a_buffer_that_the_product_reads(shmem, over, phase):
    M, N, ks, ws = 16, 1024, 1024, 4
    job = Ranks(shmem, M, N, ks, 64, 64, ws, BF16, BF16, BF16)
    on = shmem.on_rank
    for r in range(1, ws):
        job.launch(r, ops.PHASE_PRODUCE)
    torch.cuda.synchronize()
    # rank 0's operands by themselves, its result on top of one of them
    a, b = job.args[0][0].contiguous(), job.args[0][1].T.contiguous().T
    out = {"activations": a.view(M, N), "weights": b.T[:M, :].view(M, N), "partials": on(job.part, 0)}[over]
    want_part = torch.stack([O.shard_gemm(*job.shards[0], BF16)] + [on(job.part, r).cpu() for r in range(1, ws)])
    args = (a, b, on(job.part, 0), out) + job.args[0][4:]
    ops.gemm_launch(*args, phase=phase, status=job.status, partials=job.P[0], locks=job.locks[0], num_xcds=8)
    torch.cuda.synchronize()
    assert int(job.status.item()) == 0 and not on(job.flags, 0).any()
    check_close(out, O.one_shot_reduce(want_part, BF16), over)


def test_replays_of_a_graph(shmem):
    """A pass recorded once and replayed with eager work between: tiles that are signalled, and some that are not within the bound."""
    ws, M, N, ks = 8, 16, 4096, 1376
    job = Ranks(shmem, M, N, ks, 64, 64, ws, BF16, F32, BF16)
    on = shmem.on_rank
    for r in range(1, ws):
        job.launch(r, ops.PHASE_PRODUCE)
    want, late = torch.full((job.total,), ws - 1, dtype=torch.int32, device="cuda"), torch.arange(job.total, device="cuda") % 4 == 2

    def one_pass():
        on(job.flags, 0).copy_(want)
        job.launch(0, ops.PHASE_TWO_KERNELS, spin_timeout_ticks=2000)

    one_pass()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        one_pass()
    for replay in range(6):
        want.copy_(torch.where(late, ws - 2, ws - 1) if replay % 2 else torch.full_like(want, ws - 1))
        job.status.zero_()
        on(job.out, 0).fill_(-7)
        graph.replay()
        torch.cuda.synchronize()
        if replay % 2 == 0:
            job.check(0)
        else:
            assert int(job.status.item()) == 1 and not any(x.any() for x in job.locks)
            assert torch.equal(on(job.flags, 0), torch.where(late, ws - 2, 0).to(torch.int32))
