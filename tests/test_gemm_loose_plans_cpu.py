"""Which kernel is planned for operands off the 16 bytes and for a row-major B, on both sides of lines where the faster one changes
(plan names only: no GPU)."""

import pytest

from iris_amd import ops
from test_gemm_plans_cpu import F32, plan

ROWS = lambda N: dict(stride_bk=N, stride_bn=1)


@pytest.mark.parametrize("M,N,K,BM,BN,dtype,few", [
    # an odd K: rows off the 16 bytes
    (9, 4352, 12977, 256, 64, 2, False), (9, 4352, 4097, 256, 64, 2, True), (1, 4288, 32705, 128, 128, 2, False),
    (1, 3584, 23937, 256, 64, 2, True), (15, 3392, 20993, 128, 128, 2, False), (15, 1360, 19393, 128, 128, 2, True),
    (24, 5824, 449, 128, 128, 2, False), (23, 2368, 29889, 128, 128, 2, False), (24, 1600, 15489, 256, 64, 2, True),
    (36, 1376, 26745, 64, 64, 2, False), (63, 528, 27009, 64, 64, 2, True),
    # fp32, where a row of workgroups more is a round more
    (115, 6400, 10753, 128, 128, F32, False), (118, 7424, 641, 64, 64, F32, False), (118, 2368, 833, 256, 64, F32, True),
    (58, 192, 17025, 128, 128, F32, True), (40, 7552, 257, 64, 64, F32, True),
])
def test_few_rows(M, N, K, BM, BN, dtype, few):
    assert plan(M, N, K, BM, BN, dtype=dtype)[0].startswith("few_rows") == few
    # (on aligned rows the line is another)
    assert dtype == F32 or M > 16 or plan(M, N, K // 64 * 64, BM, BN)[0].startswith("few_rows")


@pytest.mark.parametrize("M,N,K,BM,BN,cells", [
    # cells that share K
    (152, 320, 29953, 128, 128, False), (209, 168, 20041, 64, 64, True), (268, 128, 19201, 64, 64, True),
    (119, 384, 17089, 128, 128, True), (66, 128, 32705, 128, 128, True), (273, 192, 16001, 128, 128, True),
])
def test_cells_that_share_k(M, N, K, BM, BN, cells):
    assert plan(M, N, K, BM, BN)[0].startswith("cells_32x32") == cells


@pytest.mark.parametrize("M,N,K,BM,BN,rows,want", [
    # operands that come from HBM: not a program per 64 x 64 part with all of K
    (83, 7936, 32384, 128, 128, True, ("128x128x64_w2x2_s4_f4_rows", 4)),
    (6745, 128, 22528, 256, 128, True, ("256x128x64_w2x2_s3_f4_rows", 9)),
    (401, 1320, 9745, 128, 128, False, ("128x128x64_w2x2_s4_f4_gather_dma", 5)),
    (73, 5824, 9281, 128, 128, False, ("128x128x64_w2x2_s4_f4_gather_dma", 5)),
    (569, 960, 3873, 256, 256, False, ("64x64x128_w2x2_s4_f4_gather_dma+parts_of_tiles", 1)),
    # cells with up to 16 rows of A
    (5, 2432, 9536, 256, 256, True, ("cells_16x32_rows", 1)),
    (2, 5696, 3840, 256, 128, True, ("cells_16x32_rows", 1)),
    (28, 4864, 7936, 64, 64, True, ("64x64x128_w2x2_s4_f4_rows", 3)),
    # a tile that is no more than half padding
    (4705, 128, 14912, 256, 256, True, ("256x128x64_w2x2_s3_f4_rows", 13)),
    (7388, 128, 22209, 256, 256, False, ("256x128x64_w2x2_s3_f4_gather_dma", 8)),
    (7388, 129, 22209, 256, 256, False, ("256x256x64_w2x4_s2_gather_dma", 8)),
])
def test_small_products(M, N, K, BM, BN, rows, want):
    assert plan(M, N, K, BM, BN, **(ROWS(N) if rows else {})) == want


@pytest.mark.parametrize("M,N,K,BM,BN,ws,partial,inside", [
    # a row-major B (K a multiple of eight)
    (2048, 2048, 128, 128, 128, 8, 2, True), (2048, 2048, 384, 128, 128, 8, 2, False), (2048, 2048, 512, 128, 128, 4, F32, True),
    (704, 7616, 128, 256, 128, 4, F32, True), (704, 7616, 128, 256, 128, 4, 2, False), (4096, 2048, 256, 256, 128, 4, F32, False),
    (3587, 448, 128, 256, 64, 4, 2, True), (3587, 448, 384, 256, 64, 4, 2, False), (3587, 448, 128, 256, 64, 8, 2, False),
    # off the 16 bytes
    (2580, 1000, 185, 256, 64, 8, 2, False), (2643, 1536, 257, 128, 128, 4, F32, True), (2643, 1536, 641, 128, 128, 8, F32, False),
    (2048, 2048, 321, 128, 128, 8, 2, True), (2048, 2048, 641, 128, 128, 8, 2, False),
    (2048, 2048, 641, 128, 128, 4, F32, True), (2048, 2048, 385, 128, 128, 8, F32, True),
    (1534, 3008, 321, 256, 128, 4, F32, True), (1534, 3008, 321, 256, 128, 4, 2, False), (4096, 2048, 321, 256, 128, 4, F32, False),
    (948, 7104, 193, 256, 256, 4, 2, False), (18, 6144, 129, 256, 64, 4, 2, True),
])
def test_reduce_inside_the_program_or_behind_it(M, N, K, BM, BN, ws, partial, inside):
    kw = ROWS(N) if K % 8 == 0 else {}
    name, _ = plan(M, N, K, BM, BN, ws=ws, epilogue=ops.EPI_ONE_SHOT, phase=ops.PHASE_FUSED, c=9 << 32, c_dtype=partial, stride_cm=N,
                   stride_cn=1, stride_cm_global=N, **kw)
    assert name.endswith("+kernel+reduce") != inside, name
