"""``matmul.apply`` under what watches a call (a trace, forward mode, torch.func, a dispatch mode): the launch in native
code must not pass it by.  What autograd's apply does there is what happens."""

import pytest
import torch
import torch.autograd.forward_ad as fwAD
from torch.utils._python_dispatch import TorchDispatchMode

from iris_amd import _native, ops
from iris_amd.matmul import matmul_all_scatter
from oracle import iris_oracle as O
from parity import check_close, make_ab

pytestmark = pytest.mark.gpu

M, N, K = 40, 64, 128


@pytest.fixture
def call(shmem):
    """(apply of (a, b, c), the published result, fresh operands on the device)."""
    cg = shmem.zeros((M, N), dtype=torch.bfloat16)
    flags = shmem.zeros((1,), dtype=torch.int32)
    bases = shmem.get_heap_bases()
    matmul_all_scatter.set_debug(False)

    def apply(a, b, c):
        return matmul_all_scatter.apply(a, b, c, cg, None, None, None, flags, 0, 1, 4, 64, 64, 64, 4, "True", 2, 8, 0, 16, 2,
                                        bases, 256)

    A, B = make_ab(M, N, K, torch.bfloat16)
    return apply, cg, (A.cuda(), B.T.contiguous().cuda().T, torch.zeros((M, N), dtype=torch.bfloat16, device="cuda"))


def native(apply, operands):
    """Whether the native code takes the call."""
    seen = []
    host = _native.host()

    class Spy:
        def __getattr__(self, name):
            return getattr(host, name)

        def matmul_apply(self, *args):
            out = host.matmul_apply(*args)
            seen.append(out is not NotImplemented)
            return out

    _native._host = Spy()
    try:
        apply(*operands)
    finally:
        _native._host = host
    return seen == [True]


def test_a_trace_holds_the_launch(call):
    apply, cg, (a, b, c) = call
    assert native(apply, (a, b, c))
    traced = torch.jit.trace(lambda a, b, c: apply(a, b, c) + 0, (a, b, c), check_trace=False)
    cg.zero_()
    A2, B2 = make_ab(M, N, K, torch.bfloat16, seed=5)
    traced(A2.cuda(), B2.T.contiguous().cuda().T, c)
    torch.cuda.synchronize()
    check_close(cg, O.shard_gemm(A2, B2, torch.bfloat16))


def test_a_tangent_is_refused(call):
    apply, cg, (a, b, c) = call
    with fwAD.dual_level():
        dual = fwAD.make_dual(a, torch.ones_like(a))
        with pytest.raises(RuntimeError, match="jvp"):
            apply(dual, b, c)


@pytest.mark.parametrize("transform", ["vmap", "jvp", "grad"])
def test_transforms_are_refused(call, transform):
    apply, cg, (a, b, c) = call

    def inside(x):  # the operands are plain tensors, the transform is around them
        apply(a, b, c)
        return x.sum()

    x = torch.ones((3, 2), device="cuda")
    cg.zero_()
    with pytest.raises(RuntimeError):
        if transform == "vmap":
            torch.func.vmap(inside)(x)
        elif transform == "jvp":
            torch.func.jvp(inside, (x,), (x,))
        else:
            torch.func.grad(inside)(x)
    torch.cuda.synchronize()
    assert not cg.any()


def test_a_dispatch_mode_sees_the_call(call):
    apply, cg, operands = call
    ops_seen = []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            ops_seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Mode():
        assert not native(apply, operands)
    torch.cuda.synchronize()
    assert cg.any() and ops_seen
    assert native(apply, operands)
    with torch.no_grad():
        assert native(apply, operands)
