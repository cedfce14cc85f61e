"""Who waits for late peers in the kernels that reduce as they store: on every shader engine a CU is left to the rank that all
others wait for, every tile that is left to another workgroup is reduced once, and the words are zero again behind it."""

import ctypes
import random

import pytest

from iris_amd import _native, ops
from test_gemm_plans_cpu import BF16, F32, plan_args

ENGINES, CUS = 32, 8  # and the CUs of an engine


def kernels(M, N, K, BM, BN, ws, phase=ops.PHASE_TWO_KERNELS, dtype=BF16, **kw):
    """(kernels, workgroups that wait at a time) of a one-shot launch"""
    kw = dict(dict(epilogue=ops.EPI_ONE_SHOT, phase=phase, c=9 << 32, stride_cm=N, stride_cn=1, stride_cm_global=N), **kw)
    n, waiting = ctypes.c_int(-1), ctypes.c_int(-1)
    args = plan_args(M, N, K, BM, BN, dtype, ws, **kw)
    assert _native.lib().iris_gemm_launch_kernels(ctypes.byref(args), ctypes.byref(n), ctypes.byref(waiting)) == 0
    return n.value, waiting.value


@pytest.mark.parametrize("ws", [2, 3, 4, 5, 7, 8, 9, 16])
def test_all_waiting_ranks_leave_room_on_every_engine(ws):
    rng, inside = random.Random(ws), 0
    for _ in range(400):
        M, N = int(2 ** rng.uniform(0, 8)), 8 * int(2 ** rng.uniform(1, 10))
        rows = dict(stride_bk=N, stride_bn=1) if rng.random() < 0.3 else {}
        n, waiting = kernels(M, N, 8 * int(2 ** rng.uniform(1, 10)), 64, rng.choice([32, 64, 128]), ws, **rows)
        if n == 1:
            inside += 1
            assert 0 < waiting and waiting * (ws - 1) <= ENGINES * (CUS - 1)
    assert (inside > 0) == (ws <= CUS)


@pytest.mark.parametrize("ws", [3, 4, 8])
def test_the_launches_that_would_fill_the_device(ws):
    # 128 tiles of two cells each, one cell a CU: with a workgroup of each tile waiting, two ranks held all CUs
    n, waiting = kernels(16, 8192, 1024, 64, 64, ws, stride_bk=8192, stride_bn=1)
    assert n == 2 or waiting * (ws - 1) <= ENGINES * (CUS - 1)
    n, waiting = kernels(16, 4096, 1376, 64, 64, ws, c_dtype=F32)
    assert n == 1 and waiting * (ws - 1) <= ENGINES * (CUS - 1)


def test_words_for_the_tiles_that_are_left():
    """Without the locks, or with all of them in use, only as many tiles as may wait on one engine are reduced inside."""
    assert kernels(16, 320, 1024, 64, 64, 8) == (1, 5)
    assert kernels(16, 16, 1024, 64, 16, 8, locks=0, partials=0) == (1, 1)
    # K shared out: the blocks of C count in the words behind the tiles', and 32 more have to be left
    for N in range(64, 4096, 64):
        n, waiting = kernels(3, N, 8192, 64, 64, 8)
        assert n == 2 or waiting <= 32


@pytest.mark.parametrize("most", [1, 2, 3, 7])
@pytest.mark.parametrize("seed", range(40))
def test_every_tile_that_is_left_is_taken_once(most, seed):
    """Workgroups in any interleaving of their accesses to memory, each the tile's last to arrive."""
    lib, rng = _native.testing_lib(), random.Random(1000 * most + seed)
    tiles = rng.choice([1, most, most + 1, 24, 128])
    word, links, done, waiting = [0], [0] * tiles, [], set()

    def swap(seen, to):
        if word[0] != seen:
            return word[0]
        word[0] = to
        return seen

    def workgroup(tile):
        seen = word[0]
        yield
        while True:
            to = lib.iris_late_join_host(seen, most, tile)
            waits = to == seen + 1
            if not waits:
                links[tile] = seen >> 8
                yield
            now = swap(seen, to)
            if now == seen:
                break
            seen = now
            if not waits:
                links[tile] = 0
            yield
        if not waits:
            return
        waiting.add(tile)
        assert len(waiting) <= most
        late = tile + 1
        while late:
            yield  # (waits, and reduces the tile)
            done.append(late - 1)
            seen = word[0]
            while True:
                late = seen >> 8
                link = links[late - 1] if late else 0
                yield
                now = swap(seen, lib.iris_late_next_host(seen, link))
                if now == seen:
                    break
                seen = now
            if late:
                links[late - 1] = 0
        waiting.discard(tile)

    running, steps = [workgroup(t) for t in range(tiles)], 0
    rng.shuffle(running)
    while running:
        # (few of them side by side, or all)
        i = rng.randrange(min(len(running), rng.choice([2, 8, 200])))
        try:
            next(running[i])
        except StopIteration:
            running.pop(i)
        steps += 1
        assert steps < 200000
    assert sorted(done) == list(range(tiles)) and word == [0] and not any(links)


@pytest.mark.parametrize("dtype", [BF16, F32])
def test_a_result_that_overlaps_what_the_product_reads_is_stored_behind_it(dtype):
    """The activations' buffer, the weights' or this rank's partials taken again for the result."""
    M, N, K, es = 16, 1024, 512, 2 if dtype == BF16 else 4
    a, b, c = 1 << 32, 2 << 32, 9 << 32
    ends = {a: M * K * es, b: N * K * es, c: M * N * es}
    result = M * N * es
    call = lambda at: kernels(M, N, K, 64, 64, 4, dtype=dtype, c_global=at)[0]  # noqa: E731
    for phase in (ops.PHASE_TWO_KERNELS, ops.PHASE_FUSED):
        assert kernels(M, N, K, 64, 64, 4, phase, dtype=dtype)[0] == 1
    for begin, size in ends.items():
        assert call(begin - result) == 1 and call(begin + size) == 1  # beside it
        assert call(begin) == 2 and call(begin - result + 16) == 2 and call(begin + size - 16) == 2
    # a row-major weight, and operands that are a part of wider ones
    assert kernels(M, N, K, 64, 64, 4, stride_bk=N, stride_bn=1, c_global=b + N * K * 2 - 16)[0] == 2
    assert kernels(M, N, K, 64, 64, 4, row=4096, c_global=a + 15 * 4096 * 2)[0] == 2
