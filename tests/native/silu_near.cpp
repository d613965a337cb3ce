// silu_near() (shield-sisa_amd/csrc/silu_near.hpp) on the CPU against x / (1 + exp(-x)) in 80 bits.  The hardware's exp2 and
// reciprocal are replaced by the correctly rounded values moved by -1, 0 and +1 ulp (both are specified to 1 ulp; subnormal
// results are flushed), every combination.  Prints the largest error in ulp over x > -16 and over the rest, and every
// limit that returns something else than the function's comment says; compiled with -ffp-contract=off as the device code is.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <limits>

static int exp_off, rcp_off;
static float moved(float v, int by) {
    for (; by > 0; --by) v = std::nextafter(v, INFINITY);
    for (; by < 0; ++by) v = std::nextafter(v, -INFINITY);
    return std::fabs(v) < std::numeric_limits<float>::min() ? std::copysign(0.0f, v) : v;
}
static float __int_as_float(int v) {
    float f;
    std::memcpy(&f, &v, 4);
    return f;
}
static int __float_as_int(float v) {
    int i;
    std::memcpy(&i, &v, 4);
    return i;
}
static float fmed3_of(float x, float lo, float hi) { return std::isnan(x) ? lo : x < lo ? lo : (x > hi ? hi : x); }
static float exp2_of(float x) { return moved(float(exp2l(x)), exp_off); }
static float rcp_of(float x) { return moved(float(1.0L / x), rcp_off); }
static float div_fixup_of(float q, float den, float num) {   // the quotient's special cases, else |q| with num / den's sign
    const float sign = std::copysign(1.0f, den) * std::copysign(1.0f, num);
    if (std::isnan(den) || std::isnan(num)) return NAN;
    if ((den == 0 && num == 0) || (std::isinf(den) && std::isinf(num))) return NAN;
    if (den == 0 || std::isinf(num)) return sign * INFINITY;
    if (std::isinf(den) || num == 0) return sign * 0.0f;
    return std::copysign(q, sign);
}
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_fmed3f fmed3_of
#define __builtin_amdgcn_exp2f exp2_of
#define __builtin_amdgcn_rcpf rcp_of
#define __builtin_amdgcn_div_fixupf div_fixup_of
#include "../../shield-sisa_amd/csrc/silu_near.hpp"

int main() {
    double upper = 0, lower = 0;
    const auto check = [&](float x) {
        const long double want = x / (1.0L + expl(-(long double)x));
        const float w = float(want);
        const double ulp = std::fabs(double(std::nextafter(w, INFINITY)) - double(w));
        const double err = std::fabs(double(shv::silu_near(x) - want)) / ulp;
        double& most = x > -16.0f ? upper : lower;
        if (err > most) most = err;
    };
    for (exp_off = -1; exp_off <= 1; ++exp_off)
        for (rcp_off = -1; rcp_off <= 1; ++rcp_off) {
            for (int i = 0; i < 200000; ++i) {
                const float t = (float(i) + 0.37f) / 200000.0f;
                check(-87.3f + 127.3f * t);          // the whole range, evenly
                check(-2.0f + 4.0f * t);
                const float s = std::exp2(-30.0f + 36.0f * t);
                if (s < 87.3f) check(-s);            // and over the logarithm
                check(s);
            }
            check(-0.693147f), check(0.346573f), check(-16.635532f), check(-16.7f), check(-24.0f);
            for (float x : {-87.5f, -88.0f, -88.6f, -89.0f, -1e4f, -3e38f}) {   // -0, where the quotient is 1e-36 at most
                const float y = shv::silu_near(x);
                if (y != 0.0f || !std::signbit(y)) std::printf("bad %g: %g\n", x, y);
            }
            for (float x : {87.5f, 200.0f, 3e38f})
                if (shv::silu_near(x) != x) std::printf("bad %g\n", x);
        }
    exp_off = rcp_off = 0;
    std::printf("%.3f %.3f\n", upper, lower);
    const float zero = shv::silu_near(0.0f), minus = shv::silu_near(-0.0f);
    if (zero != 0.0f || std::signbit(zero) || minus != 0.0f || !std::signbit(minus)) std::printf("bad zero\n");
    if (shv::silu_near(INFINITY) != INFINITY || shv::silu_near(-INFINITY) != -INFINITY) std::printf("bad infinity\n");
    if (!std::isnan(shv::silu_near(NAN)) || !std::isnan(shv::silu_near(-NAN))) std::printf("bad NaN\n");
    return 0;
}
