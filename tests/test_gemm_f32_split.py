"""The exact tier's GEMM where its K blocks go over the waves: few rows and a long K (17 to 64 K blocks of 64, up to 1,536
16 x 16 tiles), and up to 64 rows whatever the columns.  Both sides of each line, K blocks that do not divide by the four
waves, a last block of every remainder; every output the reference CPU engine's operation sequence, bit for bit."""
import pytest

import test_gemm_f32 as short_k

SHAPES = [(5, 16, 1028), (5, 384, 1100), (20, 960, 2048), (64, 40, 1284), (129, 96, 2052), (17, 17, 4096), (17, 17, 4100),
          (16, 33, 1032), (256, 1536, 1100), (257, 1536, 1100),
          (5, 30001, 64), (64, 24500, 132), (65, 24500, 132), (33, 24530, 1028)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_split_over_waves(shv, orc, weights, M, N, K):
    short_k.test_matrix_core_gemm_is_the_reference_sequence(shv, orc, weights, M, N, K)
