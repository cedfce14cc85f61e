"""Which tiles a large launch is planned in, on both sides of lines where the faster ones change (plan names only: no GPU)."""

import pytest

from test_gemm_plans_cpu import plan


@pytest.mark.parametrize("M,N,K,BM,BN,want", [
    # parts of a tile whose K would be shared out, up to some K
    (2534, 896, 1664, 256, 256, ("128x128x64_w2x2_s4_f4+parts_of_tiles", 1)),
    (1669, 320, 30872, 256, 256, ("256x256x64_w2x4_s2", 16)),
    (3319, 312, 1792, 256, 128, ("128x64x64_w2x2_s4_f4+parts_of_tiles", 1)),
    (1024, 1376, 2048, 128, 128, ("128x128x64_w2x2_s4_f4", 2)),
])
def test_parts_of_a_split_tile(M, N, K, BM, BN, want):
    assert plan(M, N, K, BM, BN) == want
