"""The exact tier's GEMM where its K blocks go over the waves: few rows and a long K (17 to 64 K blocks of 64, up to 1,536
16 x 16 tiles), and up to 64 rows whatever the columns; few outputs are the GEMV's.  Both sides of each line, K blocks that do
not divide by the four waves, a last block of every remainder; every output the reference CPU engine's operation sequence, bit
for bit."""
import numpy as np
import pytest

import test_gemm_f32 as short_k

# the last two rows: few outputs, on the GEMV and just past it
SHAPES = [(5, 16, 1028), (5, 384, 1100), (20, 960, 2048), (64, 40, 1284), (129, 96, 2052), (17, 17, 4096), (17, 17, 4100),
          (16, 33, 1032), (256, 1536, 1100), (257, 1536, 1100),
          (5, 30001, 64), (64, 24500, 132), (65, 24500, 132), (33, 24530, 1028),
          (32, 80, 960), (32, 81, 960), (64, 62, 1024), (64, 63, 768), (33, 8, 704), (32, 32, 1404), (16, 65, 1756), (8, 128, 64),
          (16, 250, 1536), (16, 251, 1536)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_split_over_waves(shv, orc, weights, M, N, K):
    short_k.test_matrix_core_gemm_is_the_reference_sequence(shv, orc, weights, M, N, K)


@pytest.mark.gpu
def test_rows_past_the_matrix_core_offsets(shv):
    """K = 2^22: past the leading dimensions that the matrix-core kernels take, the matrix-core variant included."""
    print("[gpu] gemm fp32 M=3 N=2 K=4194304", flush=True)
    hip, M, N, K = shv.Hip(), 3, 2, 1 << 22
    rng = np.random.default_rng(5)
    A, W = (rng.standard_normal((r, K), dtype=np.float32) for r in (M, N))
    dA, dW, dC = hip.upload(A), hip.upload(W), hip.malloc(M * N * 4)
    try:
        with shv.PwGemm("fp32", dW, N, K) as g:
            got = []
            for variant in (2, 0, 4):
                hip.memset(dC, 0xFF, M * N * 4)
                g.run(dA, M, dC, None, shv.ACT_NONE, variant=variant)
                hip.sync()
                got.append(hip.download(dC, (M, N), np.uint32))
        assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
        ref = A.astype(np.float64) @ W.astype(np.float64).T
        # chains of 64 products, 65,536 block sums one after another: (64 + 65536) roundings of 2^-24 of the absolute sum
        bound = (64 + K // 64) * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(W).astype(np.float64).T)
        assert (np.abs(got[0].view(np.float32) - ref) <= bound).all()
    finally:
        for p in (dA, dW, dC):
            hip.free(p)
