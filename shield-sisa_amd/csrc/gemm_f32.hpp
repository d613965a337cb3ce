// Fragments of the exact tier's matrix-core products (gemm_f32.hip, expdw.hip).
//
// Fragment layout, lane l = 16 g + r: A holds row r at k slot g, B column r at k slot g, C column r at rows 4 g ..
// 4 g + 3.  Operands are read 16 k at a time, lane (g, r) taking the float4 k = 4 g .. 4 g + 3 of row r; MFMA j of the
// chunk needs k = 4 j + g there, the 4 x 4 transpose of (lane group, element), which is two permlane32 and two
// permlane16 swaps per float4 (transpose4).
#pragma once
#include "dev_common.hpp"

namespace shv {

__device__ __forceinline__ void swap32(float& x, float& y) {   // x's upper half <-> y's lower half
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    const unsigned lo = s[0], hi = s[1];
    x = __uint_as_float(lo);
    y = __uint_as_float(hi);
}
__device__ __forceinline__ void swap16(float& x, float& y) {   // x's odd rows of 16 lanes <-> y's even rows
    const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    const unsigned lo = s[0], hi = s[1];
    x = __uint_as_float(lo);
    y = __uint_as_float(hi);
}
// lane group g, element e holds k = 4 g + e  ->  element j holds k = 4 j + g
__device__ __forceinline__ void transpose4(f32x4 v, float (&t)[4]) {
    t[0] = v[0]; t[1] = v[1]; t[2] = v[2]; t[3] = v[3];
    swap32(t[0], t[2]);
    swap32(t[1], t[3]);
    swap16(t[0], t[1]);
    swap16(t[2], t[3]);
}
__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 mfma4(float a, float w, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, w, c, 0, 0, 0);
}

}  // namespace shv
