"""The launches in native code (``csrc/host/``) against the checked Python
path behind them: same result, same errors, and what is declined."""

import pytest
import torch

from iris_amd import _native, ops, util
from iris_amd.matmul import matmul_all_scatter, matmul_one_shot_all_reduce
from oracle import iris_oracle as O
from parity import check_close, make_ab
from test_gemm_gpu import to_heap

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,workspace", [(1, True), (130, True), (130, False)])
@pytest.mark.parametrize("debug", [False, True])  # True: declined, autograd's way
def test_apply_launches_either_way(shmem, M, workspace, debug):
    N, K, ws, dtype = 200, 264, 2, torch.bfloat16
    A, B = make_ab(M, N, K, dtype)
    a, b = to_heap(shmem, A), to_heap(shmem, B)
    c = shmem.zeros((M, N), dtype=dtype)
    cg = shmem.zeros((M, N * ws), dtype=dtype)
    flags = shmem.zeros((ops.cdiv(M, 64) * ops.cdiv(N, 64),), dtype=torch.int32)
    for r in range(ws):
        shmem.on_rank(cg, r).zero_()
        shmem.on_rank(flags, r).zero_()
    P = shmem.zeros((16, 64 * 64), dtype=torch.float32) if workspace else None
    locks = shmem.zeros((16,), dtype=torch.int32) if workspace else None
    matmul_all_scatter.set_debug(debug)
    out = matmul_all_scatter.apply(a, b, c, shmem.on_rank(cg, 1), None, P, locks, shmem.on_rank(flags, 1), 1, ws, 16, 64, 64, 64, 4, "True", 2,
                                   8, 0, 16, 2, shmem.get_heap_bases(), 256)
    matmul_all_scatter.set_debug(False)
    torch.cuda.synchronize()
    assert out is not c and out.data_ptr() == c.data_ptr() and out.shape == c.shape
    for r in range(ws):
        check_close(shmem.on_rank(cg, r)[:, N:], O.shard_gemm(A, B, dtype), f"rank {r}")
        assert shmem.on_rank(flags, r).cpu().tolist() == [1] * flags.numel()


def test_what_the_native_code_declines_raises_what_it_always_did(shmem):
    a = shmem.zeros((64, 64), dtype=torch.bfloat16)
    cg = shmem.zeros((64, 64), dtype=torch.bfloat16)
    flags = shmem.zeros((1,), dtype=torch.int32)
    launch = [a, a.T, None, cg, flags, None, 0, 1, 4, 64, 64, 64, 1, ops.EPI_ALL_SCATTER]
    for at, bad, error in ((1, a.T.float(), TypeError), (3, cg[:32], ValueError), (4, flags.long(), TypeError),
                           (0, a.cpu(), RuntimeError), (13, 9, ValueError), (8, 0, ValueError)):
        args = list(launch)
        args[at] = bad
        with pytest.raises(error):
            ops.gemm_launch(*args)
    with pytest.raises(ValueError):
        ops.gemm_launch(*launch, variant=900)  # (taken, and refused by the launcher)
    host = _native.host()
    assert host.memset_i32(flags.long(), 1) == -1 and host.memset_i32(flags.cpu(), 1) == -1
    util.memset_tensor(flags, -7)
    assert flags.item() == -7
    with pytest.raises(ValueError):
        ops.one_shot_reduce(cg, cg, None, shmem.get_heap_bases(), 0, 2, 64, 64, 1)
    # an operand that wants a gradient goes through autograd
    w = a.clone().requires_grad_()
    matmul_one_shot_all_reduce.phase = ops.PHASE_TWO_KERNELS
    out = matmul_one_shot_all_reduce.apply(w, a.T, cg, cg.clone(), None, None, None, flags, 0, 1, 4, 64, 64, 64, 1, "True", 2,
                                           8, 0, 16, 2, shmem.get_heap_bases(), 256)
    matmul_one_shot_all_reduce.phase = ops.PHASE_FUSED
    assert out.requires_grad
