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


WIDE, HALF = "256x256x64_w2x4_s2", "256x128x64_w2x2_s3_f4"


@pytest.mark.parametrize("M,N,K,BM,BN,want", [
    # 256 x 64 tiles: blocks of two where a round of them does, of four where that saves rounds
    (8192, 576, 1024, 256, 64, (HALF + "+two_tiles_each", 1)),
    (8192, 704, 4096, 256, 64, (HALF + "+two_tiles_each", 1)),
    (8192, 1024, 1024, 256, 64, (HALF + "+two_tiles_each", 1)),
    (8192, 1344, 12288, 256, 64, (WIDE + "+four_tiles_each", 1)),
    # K in two parts; nine columns of tiles, the last a launch of its own
    (8192, 448, 14336, 256, 64, (HALF + "+two_tiles_each", 2)),
    (8192, 576, 36864, 256, 64, (HALF + "+two_tiles_each+last_64_columns_apart", 2)),
    # wider tiles of the caller's
    (8192, 1344, 4096, 256, 128, (WIDE + "+two_tiles_each", 1)),
    (8192, 896, 2048, 256, 128, (HALF, 1)),
    (8192, 512, 4096, 128, 128, ("128x128x64_w2x2_s4_f4", 1)),
    (855, 5120, 7872, 128, 128, (HALF + "+two_tiles_each", 1)),
    # a last round of a few tiles keeps the caller's
    (3412, 1256, 25752, 256, 64, ("256x64x64_w4x1_s3_f4+last_round_in_10_parts", 1)),
])
def test_blocks(M, N, K, BM, BN, want):
    assert plan(M, N, K, BM, BN) == want


def test_fewer_programs_than_cus_leave_none_idle():
    assert plan(1024, 640, 256, 256, 64, num_sms=16) == (HALF + "+two_tiles_each", 1)
    assert plan(1024, 640, 256, 256, 64, ws=2, num_sms=16) == (HALF + "+two_tiles_each", 1)
    assert plan(640, 392, 200, 128, 128, num_sms=8) == (HALF + "+two_tiles_each", 1)
    assert plan(1024, 640, 256, 256, 64) == ("128x64x64_w2x2_s4_f4+parts_of_tiles", 1)
