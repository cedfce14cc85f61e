"""The kernels that transpose a row-major B on its way out of LDS keep their loads in flight: a K-step waits for them where the
kernel says so and nowhere else.  (The compiler takes ds_read_b64_tr_b16 for a read that may meet any LDS-DMA it knows to be in
flight, and waits for all of it.)  From the assembly of the kernels' source: no GPU."""

import re
import subprocess

import pytest

from iris_amd import build

SOURCE = """
#include "gemm_registry.hpp"
#include "gemm_skinny.hpp"
namespace iris_amd {
IRIS_GEMM_INSTANTIATE(IRIS_DTYPE_BF16, OP_STORE16, 256, 256, 64, 2, 4, 2, LOAD_DMA_ROWS, 0, 1, "")
IRIS_GEMM_INSTANTIATE(IRIS_DTYPE_BF16, OP_STORE16, 64, 64, 128, 2, 2, 4, LOAD_DMA_ROWS, 4, 1, "")
template __global__ void gemm_skinny_kernel<IRIS_DTYPE_BF16, OP_STORE16, IRIS_DTYPE_BF16, 16, 2, 2, false, true>(const GemmKArgs);
template __global__ void gemm_skinny_kernel<IRIS_DTYPE_BF16, OP_STORE16, IRIS_DTYPE_BF16, 8, 1, 2, false, true>(const GemmKArgs);
}
"""


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{kernel: its basic blocks, lists of instructions}"""
    where = tmp_path_factory.mktemp("waits")
    (where / "kernels.hip").write_text(SOURCE)
    flags = [f for f in build.COMMON if f != "-fPIC"]
    subprocess.run([build.hipcc(), *flags, f"-I{build.CSRC}", f"-I{build.PKG.parent / 'include'}", "--cuda-device-only", "-S",
                    str(where / "kernels.hip"), "-o", str(where / "kernels.s")], check=True, capture_output=True)
    found = {}
    for text in re.split(r"\n(?=_Z\w+:)", (where / "kernels.s").read_text())[1:]:
        blocks = [[]]
        for line in text.split(".Lfunc_end")[0].splitlines()[1:]:
            if line.startswith(".LBB"):
                blocks.append([])
            elif line.startswith("\t") and line[1] not in ".;":
                blocks[-1].append(line.strip())
        found[text.split(":")[0]] = blocks
    return found


def steps(kernels, name):
    """The blocks of the kernels `name` that multiply what they have transposed."""
    blocks = [b for k, bs in kernels.items() if name in k for b in bs
              if any("ds_read_b64_tr_b16" in i for i in b) and sum("v_mfma" in i for i in b) >= 4]
    assert blocks
    return blocks


def waits_before_reads(block):
    """Waits for all loads in front of a transposing read that no barrier stands between."""
    count = pending = 0
    for i in block:
        if i.startswith("s_waitcnt") and "vmcnt(0)" in i:
            pending = 1
        elif i.startswith("s_barrier"):
            pending = 0
        elif i.startswith("ds_read_b64_tr_b16"):
            count, pending = count + pending, 0
    return count


@pytest.mark.parametrize("cm,cn", [(256, 256), (64, 64)])
def test_tiles(kernels, cm, cn):
    assert [waits_before_reads(b) for b in steps(kernels, f"gemm_persistent_kernelINS_7GemmCfgILi2ELi{cm}ELi{cn}E")
            if waits_before_reads(b)] == []


@pytest.mark.parametrize("rows", [16, 8])
def test_cells(kernels, rows):
    # (two sets in flight: the loop that refills them waits for the older one)
    loops = [b for b in steps(kernels, f"gemm_skinny_kernelILi2ELi0ELi2ELi{rows}E") if any(i.startswith("buffer_load") for i in b)]
    assert loops and all(not any("vmcnt(0)" in i for i in b) for b in loops)
