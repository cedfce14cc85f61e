"""What ``matmul.apply`` makes of the native launch's answers, with the native module replaced (no GPU)."""

import pytest
import torch

from iris_amd import _native, ops
from iris_amd.matmul import matmul_one_shot_all_reduce as matmul


class Host:
    def __init__(self, answer):
        self.answer, self.launches = answer, 0

    def matmul_apply(self, cls, epilogue, args):
        self.launches += 1
        return self.answer

    def gemm(self, *args):
        self.launches += 1
        return 0


@pytest.mark.parametrize("answer,error", [(_native.HIP_ERROR_INVALID_VALUE, ValueError), (719, RuntimeError)])
def test_a_failed_launch_is_not_made_again(monkeypatch, answer, error):
    host = Host(answer)
    monkeypatch.setattr(_native, "host", lambda: host)
    if answer != _native.HIP_ERROR_INVALID_VALUE:
        monkeypatch.setattr(_native, "hip_try", lambda err: (_ for _ in ()).throw(RuntimeError(f"HIP error code {err}")))
    t = torch.zeros(2, 2)
    with pytest.raises(error):
        matmul.apply(t, t, t, t, None, None, None, None, 0, 1, 4, 64, 64, 64, 4, "True", 2, 8, 0, 16, 2, None, 256)
    assert host.launches == 1


def test_a_declined_call_takes_the_long_way(monkeypatch):
    host = Host(NotImplemented)
    monkeypatch.setattr(_native, "host", lambda: host)
    monkeypatch.setattr(ops, "gemm_launch", lambda **kw: host.gemm())
    matmul.set_debug(False)
    t = torch.zeros(2, 2)
    out = matmul.apply(t, t, t, t, None, None, None, None, 0, 1, 4, 64, 64, 64, 4, "True", 2, 8, 0, 16, 2, None, 256)
    assert host.launches == 2 and out.data_ptr() == t.data_ptr()
    matmul.set_debug(True)
