"""Which one-shot launches reduce inside the few-rows kernel and the cells: one kernel, where a product with its reduce behind
it is two (the plan's name is the product kernel's in both)."""

import pytest

from iris_amd import ops
from test_few_rows_reduce_gpu import BF16, F16, F32, test_peers_are_done as peers_are_done
from test_late_tiles_cpu import kernels

CODE = {F32: 0, F16: 1, BF16: 2}
CASES = next(m.args[1] for m in peers_are_done.pytestmark if m.name == "parametrize" and "kernel" in m.args[0])


@pytest.mark.parametrize("M,N,ks,BM,BN,ws,dtype,part,out,rows,kernel", CASES)
@pytest.mark.parametrize("phase", [ops.PHASE_TWO_KERNELS, ops.PHASE_FUSED])
def test_the_cases_that_are_checked_on_the_gpu(M, N, ks, BM, BN, ws, dtype, part, out, rows, kernel, phase):
    kw = dict(c_dtype=CODE[part], c_global_dtype=CODE[out], scope=ops.SCOPE_SYSTEM, flag_sem=ops.FLAG_SEM_RELEASE_ACQUIRE)
    layout = dict(row=ks * ws, stride_bk=N, stride_bn=1) if rows else dict(row=ks * ws)
    if kernel.endswith("_gather_dma") and phase == ops.PHASE_FUSED:
        return  # (may be the caller's tiles, the reduce inside)
    for more in ({}, kw):
        n, waiting = kernels(M, N, ks, BM, BN, ws, phase, CODE[dtype], **dict(dict(c_dtype=CODE[part], c_global_dtype=CODE[out]), **more, **layout))
        assert n == 1 and 0 < waiting


def test_the_lines():
    one = lambda *args, **kw: kernels(*args, **kw)[0] == 1  # noqa: E731
    # tiles of a launch
    assert one(8, 128 * 16, 512, 64, 16, 2) and not one(8, 129 * 16, 512, 64, 16, 2)
    # bytes of all ranks' partials of a tile: 64 x 64 of eight is 64 KiB in 16 bits and 128 in 32; 64 x 128 of eight 256
    assert one(64, 256, 2112, 64, 64, 8) and one(64, 256, 2112, 64, 64, 8, c_dtype=0)
    assert one(64, 256, 2112, 64, 128, 8) and not one(64, 256, 2112, 64, 128, 8, c_dtype=0)
    # ranks: a wave fetches each one's strips
    assert one(8, 256, 512, 64, 64, 8) and not one(8, 256, 512, 64, 64, 9)
    # a launch that shares the device, columns that are not contiguous, timestamps
    assert not one(8, 256, 512, 64, 64, 4, num_sms=128)
    assert not one(8, 256, 512, 64, 64, 4, stride_cm_global=512, stride_cn_global=2)
    assert not one(8, 256, 512, 64, 64, 4, mm_begin_timestamp=10 << 32, mm_end_timestamp=11 << 32)
    # a product, and a reduce, of their own
    assert one(8, 256, 512, 64, 64, 4, phase=ops.PHASE_PRODUCE) and one(8, 256, 512, 64, 64, 4, phase=ops.PHASE_CONSUME)
    assert kernels(8, 256, 512, 64, 64, 4, phase=ops.PHASE_PRODUCE)[1] == 0
