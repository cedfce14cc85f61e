"""Plans of large launches whose times are as good as the same: the one by number of tiles stays (plan names only: no GPU)."""

import pytest

from test_gemm_plans_cpu import plan

LAST = "128x128x64_w2x2_s4_f4+last_round_in_%d_parts", "256x128x64_w2x2_s3_f4+last_round_in_%d_parts"


@pytest.mark.parametrize("M,N,K,BM,BN,want", [
    (1513, 8064, 35136, 256, 128, LAST[1] % 2), (2901, 4096, 13696, 256, 128, LAST[1] % 2),
    (1417, 3328, 32448, 128, 128, LAST[0] % 4), (1073, 4352, 25984, 128, 128, LAST[0] % 5),
    # ... and one that is expected to be faster by more is taken
    (8192, 704, 4096, 256, 64, "256x128x64_w2x2_s3_f4+two_tiles_each"), (8192, 1344, 12288, 256, 64, "256x256x64_w2x4_s2+four_tiles_each"),
])
def test_large(M, N, K, BM, BN, want):
    assert plan(M, N, K, BM, BN) == (want, 1)
