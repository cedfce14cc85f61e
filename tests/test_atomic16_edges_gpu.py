"""16-bit atomic accumulation at the edges of tiles and on rows that start on
an odd element: pairs of elements where both belong to the output, single ones
beside memory that does not, against the fp32-accumulated oracle."""

import pytest
import torch

from iris_amd import ops
from oracle import iris_oracle as O
from test_gemm_gpu import make_ab, to_heap

pytestmark = pytest.mark.gpu

SENTINEL = 0x7F81  # a bfloat16 that any arithmetic on it would change


@pytest.mark.parametrize("variant", [0, ops.VARIANT_PERSISTENT])
@pytest.mark.parametrize("M,N,K,BM,BN,ld,col", [
    (200, 130, 256, 128, 128, 130, 0),   # rows and columns end inside a tile, rows on even elements
    (65, 67, 192, 64, 64, 67, 0),        # rows of an odd length
    (40, 64, 2048, 64, 64, 67, 1),       # ... that start on an odd element of a wider matrix
    (1, 1, 64, 64, 64, 5, 2),
    (9, 19, 512, 16, 16, 21, 1),         # tiles of 16 columns
    (300, 72, 4608, 256, 64, 75, 3),     # K shared out
])
def test_odd_rows_and_edges(shmem, M, N, K, BM, BN, ld, col, variant):
    dtype = torch.bfloat16
    A, B = make_ab(M, N, K, dtype)
    a, b = to_heap(shmem, A), to_heap(shmem, B)
    wide = torch.full((M, ld), SENTINEL, dtype=torch.int16, device="cuda")
    whole = to_heap(shmem, wide.view(dtype))
    c = whole[:, col:col + N]
    c.zero_()
    P = shmem.zeros((256, BM * BN), dtype=torch.float32)
    locks = shmem.zeros((256,), dtype=torch.int32)
    for launch in (1, 2):
        ops.gemm_launch(a, b, None, c, None, None, 0, 1, 256, BM, BN, 64, 4, ops.EPI_ATOMIC_ADD, partials=P, locks=locks,
                        variant=variant)
        torch.cuda.synchronize()
        want = launch * O.shard_gemm(A, B, torch.float32)
        got = c.float().cpu()
        # one rounding of the product and one of the sum a launch
        assert float((got - want).abs().max()) <= 2 * launch * 2.0 ** -8 * float(want.abs().max()) + 1e-2
        bits = whole.view(torch.int16)
        assert (bits[:, :col] == SENTINEL).all() and (bits[:, col + N:] == SENTINEL).all()
