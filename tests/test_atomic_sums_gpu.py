"""Atomic launches: what an element of C is added, in which order, and what is launched for it."""

import pytest
import torch

from iris_amd import ops
from iris_amd.matmul import matmul_atomics_all_reduce
from oracle import iris_oracle as O
from parity import check_close, make_ab
from test_gemm_gather_gpu import place

pytestmark = pytest.mark.gpu

BF16, F32 = torch.bfloat16, torch.float32


def product(shmem, M, N, K):
    A, B = make_ab(M, N, K, BF16)
    a, b = place(shmem, A, False, 0, 0), place(shmem, B.T, False, 0, 0).T
    c = shmem.zeros((M, N), dtype=F32)
    return A, B, c, (a, b, None, c, None, shmem.get_heap_bases(), 0, 1, 256, 64, 64, 64, 4, ops.EPI_ATOMIC_ADD)


def kernels_of(run):
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as seen:
        run()
        torch.cuda.synchronize()
    return [e.name for e in seen.events() if "gemm" in e.name or "fill_i32" in e.name]


def test_parts_that_hand_nothing_over_need_no_locks_cleared(shmem):
    """K in parts that each add their own sums is one kernel where the library brings the workspace, too."""
    A, B, c, args = product(shmem, 266, 1152, 6248)
    assert ops.gemm_split_k(*args, num_xcds=8) > 1  # (without a workspace nothing else shares K out)
    ops.gemm_launch(*args, num_xcds=8, noalloc=True)
    torch.cuda.synchronize()
    c.zero_()
    names = kernels_of(lambda: ops.gemm_launch(*args, num_xcds=8, noalloc=True))
    assert len(names) == 1 and "gemm" in names[0], names
    check_close(c, O.shard_gemm(A, B, F32))


@pytest.mark.parametrize("M,N,K", [(266, 1152, 6248), (965, 1296, 4504)])
def test_one_sum_an_element_on_request(shmem, M, N, K):
    """split_k 1: what C held and the whole sum, rounded once, in every run; without it K of these is in parts."""
    A, B, c, args = product(shmem, M, N, K)
    P, locks = torch.zeros((256, 64 * 64), device="cuda"), torch.zeros((256,), dtype=torch.int32, device="cuda")
    assert ops.gemm_split_k(*args, num_xcds=8, partials=P, locks=locks) > 1
    assert ops.gemm_split_k(*args, num_xcds=8, partials=P, locks=locks, split_k=1) == 1

    def sums(held):
        c.fill_(held)
        matmul_atomics_all_reduce.apply(args[0], args[1], None, c, None, P, locks, None, 0, 1, 256, 64, 64, 64, 4, "True", 2, 8, 0, 16, 2,
                                        args[5], 256)
        torch.cuda.synchronize()
        return c.clone()

    matmul_atomics_all_reduce.set_debug(False)
    matmul_atomics_all_reduce.split_k = 1
    try:
        whole = sums(0.0)
        for held in (0.0, 1000.0, -0.37, 1000.0):
            assert torch.equal(sums(held), whole + held)
    finally:
        matmul_atomics_all_reduce.split_k = 0
    check_close(whole, O.shard_gemm(A, B, F32))
    check_close(sums(0.0), O.shard_gemm(A, B, F32), "in parts")
