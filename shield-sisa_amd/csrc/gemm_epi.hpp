// GEMM epilogue shared by the GEMM kernels (gemm.hip, gemm_f32.hip).
#pragma once
#include "dev_common.hpp"
#include "kernels.hpp"

namespace shv {

// out = act(v * wscale + bias) (+ residual: res 1 R + v, res 2 R + v / sqrt(2), res 3 R + 0.70710678f * v).  wscale
// is a power of two (1 unless the weight was stored pre-scaled), so v * wscale is exact.
__device__ __forceinline__ float epi_value(const GemmArgs& p, float v, float b, float res) {
    v = v * p.wscale;
    if (p.bias) v = v + b;
    v = apply_act(v, p.act);
    if (p.res == 3) v = res + 0.7071067811865475244f * v;
    else if (p.res) v = p.res == 2 ? res + v / 1.41421356237309515f : res + v;
    return v;
}
// Epilogue of the 4 x J outputs one thread holds (rows row(i), columns col(j)).  Every bias and residual operand is
// loaded (at clamped, valid addresses) before the first store: C may alias R or the bias as far as the compiler
// knows, so a load written after a store would wait for it, one memory round trip per output.
template <int J, class Row, class Col, class Val>
__device__ __forceinline__ void epi_block(const GemmArgs& p, Row row, Col col, Val val) {
    float bv[J], rv[4][J];
#pragma unroll
    for (int j = 0; j < J; ++j) bv[j] = p.bias ? p.bias[min(col(j), p.N - 1)] : 0.0f;
    if (p.res) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < J; ++j)
                rv[i][j] = p.R[min(row(i), (long long)p.M - 1) * p.ldr + min(col(j), p.N - 1)];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const long long m = row(i);
        if (m >= p.M) continue;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int n = col(j);
            if (n < p.N) p.C[m * p.ldc + n] = epi_value(p, val(i, j), bv[j], p.res ? rv[i][j] : 0.0f);
        }
    }
}

}  // namespace shv
