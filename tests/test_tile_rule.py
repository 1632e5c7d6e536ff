"""Which tiles and routes products of more than a round of tiles take (native/kernels/gemm_any.hip): priced as the kernels that run them. Rules of the host, on 256 CUs."""
from pathlib import Path

import pytest

from kgs.ops import _lib

pytestmark = pytest.mark.skipif(not Path(_lib.LIB_PATH).exists(), reason="kernels not built")


# us, read / transposed first: 48.0 / 61.9, 49.1 / 57.7, 56.2 / 66.0, 47.1 / 58.4, 67.1 / 73.3, 54.0 / 57.1, 86.3 / 90.6, 79.9 / 83.1
@pytest.mark.parametrize("M,N,K", [(3584, 11264, 384), (5120, 8192, 384), (6144, 8192, 384), (4608, 8448, 384), (7168, 8192, 384), (6400, 5888, 512), (11520, 3072, 1152),
                                   (11776, 3072, 1024)])
def test_a_k_major_operand_of_many_persistent_tiles_is_read(M, N, K):
    assert not _lib.lib().kgs_gemm_bf16_turn_b(M, N, K)


def test_a_round_costs_tiles_that_take_turns_less():
    """Rows off the 128-byte lines do not take turns above K = 1024, and their further rounds are priced so."""
    def tile(M, N, K, lda, ldb):
        t = _lib.lib().kgs_gemm_bf16_nt_tile_rows(M, N, K, lda, ldb, 0)
        return t >> 16, t & 0xffff

    for M, N, K in ((5207, 11063, 7600), (9305, 6477, 3816)):
        on, off = (K + 63) // 64 * 64, K // 64 * 64 + 72
        assert tile(M, N, K, on, on) == (256, 192) and tile(M, N, K, off, on) == tile(M, N, K, on, off) == (256, 256)
        assert tile(M, N, 1000, 1000, 1000) == tile(M, N, 1000, 1024, 1024)
    assert tile(300, 300, 64, 32, 64) == (0, 0)


# persistent / finer tile, us: 158.5 / 150.1, 97.5 / 92.4, 31.1 / 28.5, 49.3 / 46.9, 284.2 / 279.4
@pytest.mark.parametrize("M,N,K", [(2278, 11520, 3712), (2543, 10752, 2176), (2276, 12032, 384), (2033, 12800, 896), (7411, 9728, 2560)])
def test_ragged_rows_leave_the_persistent_kernel_where_finer_tiles_win(M, N, K):
    assert _lib.lib().kgs_gemm_bf16_nt_finer(M, N, K, 0, 0)
