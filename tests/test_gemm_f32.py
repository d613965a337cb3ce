"""The exact tier's GEMM on the fp32 matrix cores (gemm_f32.hip) through the C-ABI tool entry points, at the shapes where
its tiles and K blocks can go wrong: one row to past a tile, column counts around 16-column tiles and their blocks, K
below, at and past a K block with every remainder of a 16-k chunk that is a multiple of 4.

Every output is the reference CPU engine's operation sequence, so the automatic choice and the matrix-core variant
must equal the VALU tiled kernel bit for bit, and the oracle's GEMM on sampled rows."""
import numpy as np
import pytest

# (M, N, K): tiled (many rows), K blocks over waves (few rows), GEMV (<= 4 rows), the 16 -> 16 narrow layer
SHAPES = [(1, 16, 4), (4, 24, 64), (5, 24, 72), (17, 1, 12), (33, 40, 1024), (63, 100, 68), (130, 576, 384),
          (321, 384, 776), (600, 200, 80), (4097, 16, 16), (5000, 17, 24), (16385, 97, 44), (20011, 120, 40),
          (9000, 384, 1100), (40003, 72, 200)]


def operands(M, N, K, seed):
    rng = np.random.default_rng(seed)
    A = rng.standard_normal((M, K), dtype=np.float32)
    W = rng.standard_normal((N, K), dtype=np.float32)
    # rows of tiny, of signed-zero and of huge values: subnormal products, -0 sums, infinities
    A[:: 7] *= np.float32(1e-30)
    W[:: 5] *= np.float32(1e-12)
    if M > 2:
        A[1] = np.float32(-0.0)
        A[M // 2] *= np.float32(1e30)
    if N > 3:
        W[3] *= np.float32(1e10)
    b = rng.standard_normal(N, dtype=np.float32)
    return A, W, b


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_matrix_core_gemm_is_the_reference_sequence(shv, orc, weights, M, N, K):
    print(f"[gpu] gemm fp32 M={M} N={N} K={K}", flush=True)
    hip = shv.Hip()
    A, W, b = operands(M, N, K, M + N + K)
    dA, dW, db = hip.upload(A), hip.upload(W), hip.upload(b)
    out = [hip.malloc(M * N * 4) for _ in range(3)]
    try:
        with shv.PwGemm("fp32", dW, N, K) as g:
            for bias, act in ((None, shv.ACT_NONE), (db, shv.ACT_HSWISH), (db, shv.ACT_RELU)):
                got = []
                for d, variant in zip(out, (2, 0, 4)):   # tiled VALU kernel, automatic, matrix cores
                    hip.memset(d, 0xFF, M * N * 4)
                    g.run(dA, M, d, bias, act, variant=variant)
                    hip.sync()
                    got.append(hip.download(d, (M, N), np.float32))
                for what, c in zip(("automatic", "matrix cores"), got[1:]):
                    same = (c.view(np.uint32) == got[0].view(np.uint32)) | (np.isnan(c) & np.isnan(got[0]))
                    assert same.all(), f"{what}: {np.count_nonzero(~same)} of {same.size} outputs differ"
        rows = np.unique(np.linspace(0, M - 1, min(M, 40)).astype(int))
        o = orc.Oracle(weights)
        ref = o.gemm(A[rows], W, b, "relu")
        o.close()
        c = got[0][rows]
        assert ((c.view(np.uint32) == ref.view(np.uint32)) | (np.isnan(c) & np.isnan(ref))).all()
    finally:
        for p in (dA, dW, db, *out):
            hip.free(p)
