"""A call plans its launch anew each time: weighing the plans of a large launch costs little beside the one that is made."""

import ctypes
import time

import pytest

from iris_amd import _native
from test_gemm_plans_cpu import plan_args


def least_times(*calls):
    """us a call, the least of many short runs made in turn"""
    lib, parts = _native.lib(), ctypes.c_int(0)
    refs, p = [ctypes.byref(c) for c in calls], ctypes.byref(parts)
    least = [1e9] * len(calls)
    for _ in range(150):
        for i, r in enumerate(refs):
            begin = time.perf_counter()
            for _ in range(40):
                lib.iris_gemm_split_k(r, p)
            least[i] = min(least[i], (time.perf_counter() - begin) / 40 * 1e6)
    return least


@pytest.mark.parametrize("M,N,K,BM,BN,most", [
    (8192, 4096, 3584, 256, 128, 2.5), (8192, 4096, 3584, 128, 128, 2.5),
    (8192, 576, 36864, 256, 64, 6),  # (two launches)
])
def test_large(M, N, K, BM, BN, most):
    nothing, one, many = least_times(plan_args(0, N, K, BM, BN), plan_args(8192, 8192, 1024, 256, 256), plan_args(M, N, K, BM, BN))
    assert many - nothing < most * (one - nothing)
