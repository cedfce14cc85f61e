"""IRIS_FLAG_SEM_RELEASE_ACQUIRE: where several groups share a tile, the flag's release covers the last one's stores only
if every group's arrival at the tile's counter releases and acquires too.  No launch on one device can show it, so the
compiled code is looked at: each arrival has a cache write-back and an invalidate at the flag's scope of its own.  Parts of
the caller's tiles have no such arrival, and a launch whose flags are releases is not run in parts."""

import re
import shutil
import subprocess

import pytest

from iris_amd import build, ops
from test_gemm_plans_cpu import PARTS, plan

SOURCE = r"""
#include "gemm_skinny.hpp"
namespace iris_amd {
template __global__ void gemm_skinny_kernel<IRIS_DTYPE_BF16, OP_STORE16, IRIS_DTYPE_BF16, 16, 2, 2>(const GemmKArgs);
template __global__ void gemm_skinny_kernel<IRIS_DTYPE_BF16, OP_STORE16, IRIS_DTYPE_BF16, 16, 1, 1>(const GemmKArgs);
template __global__ void gemm_persistent_kernel<GemmCfg<IRIS_DTYPE_BF16, 128, 64, 64, 2, 2, 4, LOAD_DMA, 4>, OP_STORE16,
                                                IRIS_DTYPE_BF16, true>(const GemmKArgs);
}
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_arrivals_release_and_acquire(tmp_path):
    (tmp_path / "t.hip").write_text(SOURCE)
    out = tmp_path / "t.s"
    subprocess.run([build.hipcc(), *build.COMMON, "-I", str(build.CSRC), "--offload-device-only", "-S",
                    str(tmp_path / "t.hip"), "-o", str(out)], check=True, capture_output=True)
    bodies = re.split(r"^(\S+):\s*; @", out.read_text(), flags=re.M)
    kernels = {bodies[i]: bodies[i + 1].split(".Lfunc_end")[0] for i in range(1, len(bodies) - 1, 2)}
    assert len(kernels) == 3
    for name, text in kernels.items():
        for scope in ("sc1", "sc0 sc1"):  # agent, system
            arrivals = re.findall(rf"buffer_wbl2 {scope}\n(?:(?!buffer_wbl2|s_barrier).*\n)*?\s+global_atomic_add v\d+, .*\n"
                                  rf"(?:(?!buffer_wbl2|s_barrier).*\n)*?\s+buffer_inv {scope}\n", text)
            assert arrivals, (name, scope)


def test_flags_that_are_releases_are_not_raised_for_parts():
    assert plan(256, 2048, 2048, 128, 128)[0] == PARTS
    assert plan(256, 2048, 2048, 128, 128, flag_sem=ops.FLAG_SEM_RELEASE_ACQUIRE) == ("128x128x64_w2x2_s4_f4", 8)
    # (no flags, nothing to release)
    assert plan(256, 2048, 2048, 128, 128, flag_sem=ops.FLAG_SEM_RELEASE_ACQUIRE, notify=0)[0] == PARTS
