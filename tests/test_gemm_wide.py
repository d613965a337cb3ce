"""The half tiers' wide pointwise GEMM (gemm_wide_kernel) through the C-ABI tool entry points, at the shapes where its
pairs of column tiles and its weight registers can go wrong: odd tile counts, a last tile of 4 columns, groups of two and
of four tiles, one K step to eight, K steps cut short, rows below, at and past a workgroup's 64.

Every MFMA kernel variant performs the same operations per output, so the wide kernel and the automatic choice must equal
the direct kernel (one column tile per wave) bit for bit."""
import numpy as np
import pytest

SHAPES = [(1, 4, 8), (63, 180, 40), (64, 192, 64), (65, 196, 72), (130, 336, 96), (2049, 184, 160), (2113, 960, 152),
          (3000, 260, 192), (8200, 212, 200), (8257, 480, 256), (700, 20, 248)]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("mode", ["fp16", "bf16"])
def test_wide_gemm_equals_direct(shv, mode, M, N, K):
    if mode == "bf16" and K > 192:
        pytest.skip("bf16 takes K <= 192 here")
    print(f"[gpu] gemm wide {mode} M={M} N={N} K={K}", flush=True)
    hip = shv.Hip()
    rng = np.random.default_rng(M + N + K)
    A = rng.standard_normal((M, K), dtype=np.float32)
    W = rng.standard_normal((N, K), dtype=np.float32)
    dA, dW, db = hip.upload(A), hip.upload(W), hip.upload(rng.standard_normal(N, dtype=np.float32))
    out = [hip.malloc(M * N * 4) for _ in range(3)]
    try:
        with shv.PwGemm(mode, dW, N, K) as g:
            for bias, act in ((None, shv.ACT_NONE), (db, shv.ACT_HSWISH)):
                got = []
                for d, variant in zip(out, (2, 9, 0)):   # direct, wide, automatic
                    hip.memset(d, 0xFF, M * N * 4)
                    g.run(dA, M, d, bias, act, variant=variant)
                    hip.sync()
                    got.append(hip.download(d, (M, N), np.float32).view(np.uint32))
                assert np.array_equal(got[1], got[0]), "wide kernel"
                assert np.array_equal(got[2], got[0]), "automatic choice"
        ref = A.astype(np.float64) @ W.astype(np.float64).T
        bound = 2.0 ** -17 * (np.abs(A).astype(np.float64) @ np.abs(W).astype(np.float64).T)   # split operands
        with shv.PwGemm(mode, dW, N, K) as g:
            g.run(dA, M, out[0], None, shv.ACT_NONE, variant=9)
            hip.sync()
        assert (np.abs(hip.download(out[0], (M, N), np.float32) - ref) <= bound).all()
    finally:
        for p in (dA, dW, db, *out):
            hip.free(p)
