// SiLU of the SHIELD-A blocks.  Nothing but builtins, so that the function can be compiled and checked on the CPU with
// stand-ins for them.
#pragma once

namespace shv {

// x / (1 + exp(-x)) in 16 instructions (silu() and the libm form take 35 to 45).  exp(-x) = 2^n 2^f by Cody and Waite's
// reduction (log2 e in two parts) and the hardware exp2 of the fraction; 1 + exp(-x) as the sum d and its rounding error dl
// (Dekker's Fast2Sum, exact up to exp(-x) = 2^24; beyond, for x < -16.6, dl may be one off, an ulp of d at most); the quotient
// by the hardware reciprocal and one residual step against d + dl.  At most 3.5 ulp off for x > -16 and 4.5 down to -87.3
// were the hardware's exp2 and reciprocal an ulp off everywhere.  On the device, against 64 bits, it is at most 1.8 and 2.8
// ulp off (silu() 2.0 and 2.5, the libm form 2.1 and 2.8), and over 4 M normal x of scale 0.01 to 5 its relative error
// (2-norm) is 2.5e-8 to 2.9e-8 (silu() and the libm form 4.0e-8 to 4.4e-8), its mean 0.28 to 0.29 ulp (0.37 to 0.42).
// Limits: the reciprocal of more than 2^126 is zero, so below -87.3 the result is -0 (the libm form: about -1e-36 down to
// -88.7, then -0), and exp's argument is clamped there, so that -inf gives -inf, as silu()'s clamp does (the libm form: NaN);
// +inf gives +inf, NaN stays NaN and zeros keep their sign (div_fixup).
__device__ __forceinline__ float silu_near(float x) {
    constexpr float MAGIC = 12582912.0f;   // 1.5 * 2^23: its sum with |y| < 2^22 holds rint(y) in the low bits
    const float c = __builtin_amdgcn_fmed3f(x, -87.4f, 87.0f);
    const float m = __builtin_fmaf(c, -1.44269504088896341f, MAGIC), n = m - MAGIC;
    float f = __builtin_fmaf(c, -1.44269504088896341f, -n);
    f = __builtin_fmaf(c, -1.92596299e-8f, f);
    const float e = __int_as_float(__float_as_int(__builtin_amdgcn_exp2f(f)) + (__float_as_int(m) << 23));
    const float d = 1.0f + e, dl = e - (d - 1.0f), r = __builtin_amdgcn_rcpf(d);
    float q = x * r;
    q = __builtin_fmaf(__builtin_fmaf(-dl, q, __builtin_fmaf(-d, q, x)), r, q);
    return __builtin_amdgcn_div_fixupf(q, d, x);
}

}  // namespace shv
