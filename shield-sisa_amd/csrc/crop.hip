// Face crops on the GPU: the reference's lazy native crop (engine/preprocess/canvas.cpp:66-91, shv_prep.h:181-186)
//   crop = cv2.resize(canvas[4y:4(y+h), 4x:4(x+w)], (320, 180), INTER_AREA)
// where canvas is the native frame resized into 1280x720 (INTER_AREA when shrinking, INTER_LINEAR when enlarging,
// letterbox bars zero; engine/preprocess/geometry.cpp:77-88).  Every output byte is a fixed function of a small
// source neighbourhood.  One kernel: a workgroup walks down a band of a crop's output rows, computing the canvas rows
// that the next one needs (only those) into LDS and resizing them from there, so no canvas pixel reaches HBM.
//
// The resize arithmetic is OpenCV 4.13's for 8-bit images, as the reference restates it in
// engine/preprocess/cvresize.cpp:
//   area, general scale (cvresize.cpp:22-38, 303-335, 421-447): per output, for each source row of its area tab in
//     order: t = ((0 + S0 a0) + S1 a1) + ... over the column taps, sum = b0 t0 (first row) then sum + b_j t_j;
//     out = saturate(rint(sum)); every float operation rounded separately;
//   area, integer scale (cvresize.cpp:612-666): 2x2 blocks (S00 + S01 + S10 + S11 + 2) >> 2, other full blocks
//     rint((float)sum * (1.f / (ix iy))) (the source is a whole number of blocks at an integer scale);
//   linear, 11-bit fixed point (cvresize.cpp:185-212, 668-719): h = S[x] a0 + S[x+1] a1 (or S[x] 2048 past lxmax),
//     out = (((b0 (h0 >> 4)) >> 16) + ((b1 (h1 >> 4)) >> 16) + 2) >> 2, rows clipped into the source;
//   equal sizes: copy.
// All four are one row pass and one column pass here, over K x K source pixels per output.  The row pass is
// t = S0 w0 + S1 w1 + ... in fp32: the area weights; 1 for a block and the copy; the 11-bit coefficients (sums below
// 2^24, exact).  The column pass adds the K rows' t with their weights and finishes by kind.  Taps that an output does
// not have are zero weights: t + 0 is t.
// The plan tables (taps, weights, coefficients) are built on the host in the reference's double / float arithmetic.
// I420 frames are converted per native pixel as the reference does row by row (engine/preprocess/color.cpp:4-11,
// 57-109: ffmpeg's unscaled yuv420p -> rgb24, BT.601 limited range, 16-bit fixed point, chroma of (x, y) at
// [y / 2][x / 2]).
#include "crop_plan.hpp"
#include "dev_common.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <array>
#include <cstring>
#include <map>
#include <mutex>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

namespace shv {
namespace {

#define CROP_CHECK(expr)                                                                                     \
    do {                                                                                                     \
        const hipError_t err__ = (expr);                                                                     \
        if (err__ != hipSuccess) throw std::runtime_error(std::string("HIP error ") + hipGetErrorString(err__)); \
    } while (0)

constexpr int CROP_RING = 6;    // canvas rows in LDS: an output row takes at most five
static_assert(CROP_RING > CROP_KMAX, "an output row's canvas rows and the ring");

// one resize geometry on the device.  Output column x reads the K source pixels from xoff[x] with weights xw[x * K ..];
// output row y the source rows ysi[y * K ..] with weights yw[y * K ..].  fin: how a column pass ends.
struct PlanDev {
    int fin = FIN_SCALE, K = 1, sw = 0, sh = 0;
    float fscale = 1.0f;
    const int *xoff = nullptr, *ysi = nullptr;
    const float *xw = nullptr, *yw = nullptr;
};

// The job and plan tables hold generic pointers; these say that they are global (vector loads without the LDS aperture
// check) and, for the per-row tables, read-only and uniform (scalar loads).
#define AS_GLOBAL __attribute__((address_space(1)))
#define AS_CONST __attribute__((address_space(4)))
typedef const AS_GLOBAL uint8_t* GBytes;
typedef unsigned UWord __attribute__((aligned(1)));
__device__ __forceinline__ GBytes global_bytes(const uint8_t* p) { return (GBytes)p; }

// one crop: its native frame, canvas geometry and patch
struct JobDev {
    const uint8_t* frame;   // RGB, or the I420 Y plane
    long long stride;
    const uint8_t *u, *v;   // I420 chroma planes
    long long u_stride, v_stride;
    int canvas_plan, crop_plan;
    int px0, py0, pw, ph;  // patch = canvas columns px0 .. px0+pw, rows py0 .. py0+ph
    int left, top, new_w, new_h;
    int index;             // of the crop in the output
};

// saturate(rint(v)) (cvRound: round half to even) into byte c of o
__device__ __forceinline__ unsigned put_u8(float v, int c, unsigned o) {
    return __builtin_amdgcn_cvt_pk_u8_f32(__builtin_amdgcn_fmed3f(__builtin_rintf(v), 0.0f, 255.0f), c, o);
}
// byte i of consecutive little-endian words (i is a compile-time constant after unrolling)
__device__ __forceinline__ unsigned byte_of(const unsigned* w, int i) { return (w[i >> 2] >> (8 * (i & 3))) & 255u; }

// N bytes from p on as words, at any address; up to three bytes more are read
template <int N> __device__ __forceinline__ void load_bytes(GBytes p, unsigned (&w)[load_words(N)]) {
#pragma unroll
    for (int d = 0; d < load_words(N); ++d) w[d] = *reinterpret_cast<const AS_GLOBAL UWord*>(p + 4 * d);
}

__device__ __forceinline__ void yuv_px(int y, int u, int v, float (&o)[3]) {
    const int yy = yuv_luma(y);
    o[0] = float(yuv_sat8(yy + yuv_red(v)));
    o[1] = float(yuv_sat8(yy + yuv_green(u, v)));
    o[2] = float(yuv_sat8(yy + yuv_blue(u)));
}

// Native sources.  Row: where a source row starts (uniform).  Raw<K>: what a thread loads of a row for K pixels from
// column x on, in words (crop_variant() says why the bytes past them are there; `last`: the rows read byte by byte);
// tap(): pixel k of them.
struct RgbSrc {
    GBytes f;
    long long stride;
    int h;
    struct Row { GBytes p; };
    template <int K> struct Raw { unsigned px[load_words(3 * K)]; };
    __device__ bool last(int y) const { return y == h - 1; }
    __device__ Row row(int y) const { return {f + (long long)y * stride}; }
    template <int K> __device__ void load(int x, const Row& q, Raw<K>& r) const { load_bytes<3 * K>(q.p + unsigned(3 * x), r.px); }
    template <int K> __device__ void tap(const Raw<K>& r, int, int k, float (&o)[3]) const {
#pragma unroll
        for (int c = 0; c < 3; ++c) o[c] = float(byte_of(r.px, 3 * k + c));
    }
    __device__ void pixel(int x, const Row& q, float (&o)[3]) const {
#pragma unroll
        for (int c = 0; c < 3; ++c) o[c] = float(q.p[unsigned(3 * x) + c]);
    }
};
struct I420Src {   // converted per pixel
    GBytes Y, U, V;
    long long ys, us, vs;
    int h;
    struct Row { GBytes y, u, v; };
    template <int K> struct Raw { unsigned y[load_words(K)], u[load_words(chroma_samples(K))], v[load_words(chroma_samples(K))]; };
    __device__ bool last(int y) const { return (y >> 1) == ((h + 1) >> 1) - 1; }
    __device__ Row row(int y) const {
        return {Y + (long long)y * ys, U + (long long)(y >> 1) * us, V + (long long)(y >> 1) * vs};
    }
    template <int K> __device__ void load(int x, const Row& q, Raw<K>& r) const {
        constexpr int C = chroma_samples(K);
        load_bytes<K>(q.y + unsigned(x), r.y);
        load_bytes<C>(q.u + (unsigned(x) >> 1), r.u);
        load_bytes<C>(q.v + (unsigned(x) >> 1), r.v);
    }
    template <int K> __device__ void tap(const Raw<K>& r, int x, int i, float (&o)[3]) const {
        const int odd = x & 1;
        const auto chroma = [&](const unsigned* c) {
            if constexpr (load_words(chroma_samples(K)) == 1) return (c[0] >> (8 * ((i + odd) >> 1))) & 255u;
            return odd ? byte_of(c, (i + 1) >> 1) : byte_of(c, i >> 1);
        };
        yuv_px(int(byte_of(r.y, i)), int(chroma(r.u)), int(chroma(r.v)), o);
    }
    __device__ void pixel(int x, const Row& q, float (&o)[3]) const {
        yuv_px(q.y[unsigned(x)], q.u[unsigned(x) >> 1], q.v[unsigned(x) >> 1], o);
    }
};
struct RingSrc {   // canvas rows in the LDS ring, one word (R, G, B) per pixel
    const unsigned* px;
    int width;   // of a row
    struct Row { const unsigned* p; };
    template <int K> struct Raw { unsigned px[K]; };
    __device__ Row row(int y) const { return {px + (y % CROP_RING) * width}; }
    template <int K> __device__ void load(int x, const Row& q, Raw<K>& r) const {
#pragma unroll
        for (int k = 0; k < K; ++k) r.px[k] = q.p[x + k];
    }
    template <int K> __device__ void tap(const Raw<K>& r, int, int k, float (&o)[3]) const {
#pragma unroll
        for (int c = 0; c < 3; ++c) o[c] = float(byte_of(r.px + k, c));
    }
};

// The column pass: rows' t in order, then the finish: R | G << 8 | B << 16.
template <int FIN> struct Column {
    float sum[3];
    int acc[3];
    __device__ __forceinline__ void add(bool first, float b, const float (&t)[3]) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if constexpr (FIN == FIN_LINEAR) {
                const int v = (int(b) * (int(t[c]) >> 4)) >> 16;
                acc[c] = first ? v : acc[c] + v;
            } else {
                const float bt = b * t[c];
                sum[c] = first ? bt : sum[c] + bt;
            }
        }
    }
    __device__ __forceinline__ unsigned finish(float fscale) const {
        unsigned o = 0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if constexpr (FIN == FIN_QUARTER) o |= unsigned((int(sum[c]) + 2) >> 2) << (8 * c);
            else if constexpr (FIN == FIN_LINEAR) o |= unsigned((acc[c] + 2) >> 2) << (8 * c);
            else o = put_u8(sum[c] * fscale, c, o);
        }
        return o;
    }
};
// the source rows of one output row and their weights (all uniform)
template <int K, class Src> struct Rows {
    typename Src::Row row[K];
    float b[K];
    __device__ __forceinline__ Rows(const PlanDev& p, const Src& src, int y) {
#pragma unroll
        for (int j = 0; j < K; ++j) {
            row[j] = src.row(((const AS_CONST int*)p.ysi)[y * K + j]);
            b[j] = ((const AS_CONST float*)p.yw)[y * K + j];
        }
    }
};
// the row pass of K pixels
template <int K, class Src>
__device__ __forceinline__ void row_pass(const Src& src, const typename Src::template Raw<K>& raw, int x0, const float* w,
                                         float (&t)[3]) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
        float v[3];
        src.template tap<K>(raw, x0, k, v);
#pragma unroll
        for (int c = 0; c < 3; ++c) t[c] = k == 0 ? v[c] * w[k] : t[c] + v[c] * w[k];
    }
}
// one output pixel of those rows: first source column x0, column weights w
template <int K, int FIN, class Src>
__device__ __forceinline__ unsigned resize_px(const Rows<K, Src>& rows, const Src& src, int x0, const float* w, float fscale) {
    Column<FIN> col;
    typename Src::template Raw<K> raw[K];
#pragma unroll
    for (int j = 0; j < K; ++j) src.template load<K>(x0, rows.row[j], raw[j]);
#pragma unroll
    for (int j = 0; j < K; ++j) {
        float t[3];
        row_pass<K>(src, raw[j], x0, w, t);
        col.add(j == 0, rows.b[j], t);
    }
    return col.finish(fscale);
}
// the same for wide K, two rows at a time (all of them at once took up to 243 registers)
template <int K, int FIN, class Src>
__device__ __forceinline__ unsigned resize_px_wide(const PlanDev& p, const Src& src, int y, int x0, const float* w) {
    Column<FIN> col;
#pragma unroll 2
    for (int j = 0; j < K; ++j) {
        typename Src::template Raw<K> raw;
        src.template load<K>(x0, src.row(((const AS_CONST int*)p.ysi)[y * K + j]), raw);
        float t[3];
        row_pass<K>(src, raw, x0, w, t);
        col.add(j == 0, ((const AS_CONST float*)p.yw)[y * K + j], t);
    }
    return col.finish(p.fscale);
}
// output pixel (x, y) of any plan, source pixel by source pixel, all inside the source; x and y may differ by thread
template <int UNROLL, int FIN, class Src>
__device__ __forceinline__ unsigned resize_any_fin(const PlanDev& p, const Src& src, int x, int y) {
    const auto xw = (const AS_GLOBAL float*)p.xw + x * p.K;
    const auto ysi = (const AS_GLOBAL int*)p.ysi + y * p.K;
    const auto yw = (const AS_GLOBAL float*)p.yw + y * p.K;
    const int x0 = ((const AS_GLOBAL int*)p.xoff)[x];
    Column<FIN> col;
    for (int j = 0; j < p.K; ++j) {
        const typename Src::Row row = src.row(ysi[j]);
        float t[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll UNROLL
        for (int k = 0; k < p.K; ++k) {
            float v[3];
            src.pixel(min(x0 + k, p.sw - 1), row, v);
            const float a = xw[k];
#pragma unroll
            for (int c = 0; c < 3; ++c) t[c] = t[c] + v[c] * a;
        }
        col.add(j == 0, yw[j], t);
    }
    return col.finish(p.fscale);
}
template <int UNROLL, class Src> __device__ __forceinline__ unsigned resize_any(const PlanDev& p, const Src& src, int x, int y) {
    switch (p.fin) {
    case FIN_QUARTER: return resize_any_fin<UNROLL, FIN_QUARTER>(p, src, x, y);
    case FIN_LINEAR: return resize_any_fin<UNROLL, FIN_LINEAR>(p, src, x, y);
    default: return resize_any_fin<UNROLL, FIN_SCALE>(p, src, x, y);
    }
}

constexpr int CROP_THREADS = CROP_W, CROP_PASS = 1280 / CROP_THREADS;   // canvas columns per thread

// The patch columns of a workgroup: pa .. pb in the ring, of which la .. lb lie on the frame and the others under its
// letterbox bars (zero in every ring row, written once).
struct Span {
    int pa, pb, la, lb;
    __device__ int width() const { return pb - pa; }
    __device__ int live() const { return lb - la; }
};
// A thread's (up to four) live columns' taps, kept for the whole band.
template <int K> struct Columns {
    int x0[CROP_PASS];
    float w[CROP_PASS][K ? K : 1];
};
// Canvas rows ya .. yb - 1 of the patch into the ring.
template <int K, int FIN, class Src>
__device__ __forceinline__ void fill_rows(const JobDev& j, const PlanDev& p, const Src& src, const Columns<K>& cs,
                                          const Span& sp, int ya, int yb, unsigned* ring) {
    const int live = sp.live(), xa = j.px0 + sp.la - j.left;   // column of the resized frame of the first live one
    if (live <= 0) return;
    unsigned* base = ring + (sp.la - sp.pa);
    if constexpr (K == 0) {   // rows and columns together: few of them may be live
        for (int i = threadIdx.x; i < (yb - ya) * live; i += CROP_THREADS) {
            const int r = ya + i / live, px = i % live, y = r + j.py0 - j.top;
            base[(r % CROP_RING) * sp.width() + px] = y >= 0 && y < j.new_h ? resize_any<4>(p, src, xa + px, y) : 0u;
        }
        return;
    }
    for (int r = ya; r < yb; ++r) {
        const int y = r + j.py0 - j.top;   // row of the resized frame; outside it the letterbox bars
        unsigned* row = base + (r % CROP_RING) * sp.width();
        const bool bar = y < 0 || y >= j.new_h;
        if (!bar && !src.last(((const AS_CONST int*)p.ysi)[y * p.K + p.K - 1])) {
            if constexpr (K > 0) {
                // uniform passes; a column past the last live one is computed (from its clamp) and dropped
                const auto passes = [&](auto pixel) {
#pragma unroll
                    for (int q = 0; q < CROP_PASS; ++q) {
                        if (CROP_THREADS * q >= live) break;
                        const int px = threadIdx.x + CROP_THREADS * q;
                        const unsigned v = pixel(cs.x0[q], cs.w[q]);
                        if (px < live) row[px] = v;
                    }
                };
                if constexpr (K <= CROP_KMAX) {
                    const Rows<K, Src> rows(p, src, y);
                    passes([&](int x0, const float* w) { return resize_px<K, FIN>(rows, src, x0, w, p.fscale); });
                } else {
                    passes([&](int x0, const float* w) { return resize_px_wide<K, FIN>(p, src, y, x0, w); });
                }
            }
        } else {
            for (int px = threadIdx.x; px < live; px += CROP_THREADS) row[px] = bar ? 0u : resize_any<1>(p, src, xa + px, y);
        }
    }
}
// the four pixels of a lane quad as three words: word i = the last 3 - i bytes of pixel i and the first i + 1 of the next
__device__ __forceinline__ unsigned quad_word(unsigned px, int i) {
    const unsigned next = unsigned(__builtin_amdgcn_update_dpp(0, int(px), 0xF9, 0xf, 0xf, false));   // quad_perm 1,2,3,3
    return (px >> (8 * i)) | (next << (24 - 8 * i));
}

// one output pixel per thread from the ring, for the crop plan's K (1 .. 5) and finish
template <int K, int FIN>
__device__ __forceinline__ unsigned out_px(const PlanDev& p, const RingSrc& src, int x0, const float (&w)[CROP_KMAX], int y) {
    return resize_px<K, FIN>(Rows<K, RingSrc>(p, src, y), src, x0, w, p.fscale);
}
__device__ __forceinline__ unsigned out_px_any(const PlanDev& p, const RingSrc& src, int x0, const float (&w)[CROP_KMAX], int y) {
    switch (p.K) {   // uniform
    case 1: return out_px<1, FIN_SCALE>(p, src, x0, w, y);
    case 2:
        return p.fin == FIN_QUARTER ? out_px<2, FIN_QUARTER>(p, src, x0, w, y) : out_px<2, FIN_SCALE>(p, src, x0, w, y);
    case 3: return out_px<3, FIN_SCALE>(p, src, x0, w, y);
    case 4: return out_px<4, FIN_SCALE>(p, src, x0, w, y);
    default: return out_px<5, FIN_SCALE>(p, src, x0, w, y);
    }
}

template <int K, int FIN, class Src>
__device__ __forceinline__ void crop_band(const JobDev& j, const PlanDev& np, const PlanDev& cp, const Src& src, int oy0,
                                          int oy1, int oc0, int cols, unsigned* ring, uint8_t* out) {
    const auto cxoff = (const AS_CONST int*)cp.xoff;
    Span sp;
    sp.pa = cxoff[oc0];
    sp.pb = cxoff[oc0 + cols - 1] + cp.K;
    sp.la = max(sp.pa, j.left - j.px0);
    sp.lb = min(sp.pb, j.left + j.new_w - j.px0);
    if (sp.live() < sp.width()) {
        const int width = sp.width();
        for (int i = threadIdx.x; i < CROP_RING * width; i += CROP_THREADS) {
            const int px = sp.pa + i % width;
            if (px < sp.la || px >= sp.lb) ring[i] = 0u;
        }
    }
    Columns<K> cs;
#pragma unroll
    for (int q = 0; q < CROP_PASS; ++q) {
        const int px = sp.la + min(int(threadIdx.x) + CROP_THREADS * q, max(sp.live() - 1, 0));
        const int x = min(max(j.px0 + px - j.left, 0), j.new_w - 1);
        cs.x0[q] = ((const AS_GLOBAL int*)np.xoff)[x];
#pragma unroll
        for (int k = 0; k < K; ++k) cs.w[q][k] = ((const AS_GLOBAL float*)np.xw)[x * K + k];
    }
    const int ox = oc0 + min(int(threadIdx.x), cols - 1);
    const int ox0 = ((const AS_GLOBAL int*)cp.xoff)[ox] - sp.pa;
    float ow[CROP_KMAX];
#pragma unroll
    for (int k = 0; k < CROP_KMAX; ++k) ow[k] = k < cp.K ? ((const AS_GLOBAL float*)cp.xw)[ox * cp.K + k] : 0.0f;
    const auto ysi = (const AS_CONST int*)cp.ysi;
    const RingSrc rs{ring, sp.width()};
    const bool words = (reinterpret_cast<uintptr_t>(out) & 3) == 0, mine = int(threadIdx.x) < cols;
    uint8_t* d = out + 3 * CROP_W * oy0;
    int have = ysi[oy0 * cp.K];   // patch rows below this one are in the ring (or not needed)
    for (int oy = oy0; oy < oy1; ++oy, d += 3 * CROP_W) {
        const int need = ysi[oy * cp.K + cp.K - 1] + 1;
        fill_rows<K, FIN>(j, np, src, cs, sp, have, need, ring);
        have = max(have, need);
        __syncthreads();
        const unsigned v = out_px_any(cp, rs, ox0, ow, oy);
        if (words) {   // cols is a multiple of four: a lane quad is in or out
            const int i = ox & 3;
            const unsigned w = quad_word(v, i);
            if (mine && i < 3) *reinterpret_cast<unsigned*>(d + 3 * (ox - i) + 4 * i) = w;
        } else if (mine) {
            d[3 * ox] = uint8_t(v);
            d[3 * ox + 1] = uint8_t(v >> 8);
            d[3 * ox + 2] = uint8_t(v >> 16);
        }
        __syncthreads();   // the next rows go into slots that this row's threads may still read
    }
}

// Workgroup (band of output rows and chunk of their columns, crop) of five waves: per output row the canvas rows it adds
// (each thread its columns, so a wave reads neighbouring pixels), then one output pixel per thread.  Reads the native pixels
// under a crop once (a row or two more per band) and writes the crop; bound by the instructions of the row pass for many
// crops (a conversion, a product and a sum per byte and tap; VALU 60% busy at 640 crops, four waves a SIMD, 2.1 TB/s), by a
// workgroup's rows one after another for few.
// Kernel time of 640 crops of 1920 x 1080 RGB frames 1.10 ms, of 80 crops of 1280 x 720 I420 frames 150 us; the calls 6.44 ->
// 1.51 ms and 414 -> 197 us (two kernels, canvas patches through HBM, tap loops over byte loads before).
template <bool I420, int V>
__global__ void __launch_bounds__(CROP_THREADS)
crop_kernel(const JobDev* __restrict__ jobs, const PlanDev* __restrict__ plans, uint8_t* __restrict__ out,
            int band, int chunks) {
    extern __shared__ __attribute__((aligned(16))) unsigned ring[];
    constexpr int K = kVariants[V].K, FIN = kVariants[V].fin;
    const JobDev j = jobs[blockIdx.y];
    const int cols = CROP_W / chunks, oc0 = int(blockIdx.x % chunks) * cols;
    const int oy0 = int(blockIdx.x / chunks) * band, oy1 = min(CROP_H, oy0 + band);
    const PlanDev cp = plans[j.crop_plan], np = plans[j.canvas_plan];
    uint8_t* d = out + (long long)j.index * (CROP_W * CROP_H * 3);
    if constexpr (I420) {
        const I420Src src{global_bytes(j.frame), global_bytes(j.u), global_bytes(j.v), j.stride, j.u_stride, j.v_stride,
                          np.sh};
        crop_band<K, FIN>(j, np, cp, src, oy0, oy1, oc0, cols, ring, d);
    } else {
        const RgbSrc src{global_bytes(j.frame), j.stride, np.sh};
        crop_band<K, FIN>(j, np, cp, src, oy0, oy1, oc0, cols, ring, d);
    }
}

// Plans uploaded once per geometry; the device plan table and the job tables grow as needed.  One call at a time.
class CropEngine {
public:
    static CropEngine& get() {
        static CropEngine e;
        return e;
    }
    void run(const CropJob* jobs, int n, uint8_t* out, hipStream_t s, bool i420) {
        // every argument is checked before the device is touched
        std::vector<CanvasGeo> geo(static_cast<size_t>(n));
        for (int i = 0; i < n; ++i) {
            const CropJob& j = jobs[i];
            if (!j.frame || j.width <= 0 || j.height <= 0 || j.stride < (i420 ? 1LL : 3LL) * j.width ||
                (i420 && (!j.u || !j.v || j.u_stride < (j.width + 1) / 2 || j.v_stride < (j.width + 1) / 2)))
                throw std::runtime_error("crops: bad frame " + std::to_string(i));
            if (j.x < 0 || j.y < 0 || j.w <= 0 || j.h <= 0 || j.x + j.w > CROP_W || j.y + j.h > CROP_H)
                throw std::runtime_error("crops: rect out of the 320x180 letterbox at crop " + std::to_string(i));
            if (4 * j.w < CROP_W || 4 * j.h < CROP_H)
                throw std::runtime_error("crops: rect smaller than 80x45 (no INTER_AREA shrink) at crop " +
                                         std::to_string(i));
            if (!canvas_geo(j.width, j.height, geo[size_t(i)])) throw std::runtime_error("crops: frame size");
        }
        std::lock_guard<std::mutex> lk(mu_);
        int dev = 0;
        CROP_CHECK(hipGetDevice(&dev));
        if (device_ >= 0 && dev != device_) throw std::runtime_error("crops: one device per process");
        device_ = dev;
        grow_host(jobs_host_, jobs_host_bytes_, size_t(n) * sizeof(JobDev));
        JobDev* jd = static_cast<JobDev*>(jobs_host_);
        std::vector<JobDev> all(static_cast<size_t>(n));
        std::vector<int> kn(static_cast<size_t>(n));
        // per variant: crops, widest patch, widest resized frame
        int first[CROP_VARIANTS + 1] = {}, patch_w[CROP_VARIANTS] = {}, frame_w[CROP_VARIANTS] = {};
        for (int i = 0; i < n; ++i) {
            const CropJob& j = jobs[i];
            const CanvasGeo& g = geo[size_t(i)];
            JobDev& d = all[size_t(i)];
            d.frame = j.frame;
            d.stride = j.stride;
            d.u = j.u; d.v = j.v; d.u_stride = j.u_stride; d.v_stride = j.v_stride;
            d.canvas_plan = plan_index({0, j.width, j.height, g.new_w, g.new_h, g.mode == 2 ? 1 : 3});
            d.crop_plan = plan_index({1, 4 * j.w, 4 * j.h, CROP_W, CROP_H, 3});
            d.px0 = 4 * j.x; d.py0 = 4 * j.y; d.pw = 4 * j.w;
            d.left = g.left; d.top = g.top; d.new_w = g.new_w; d.new_h = g.new_h;
            d.index = i;
            if (plans_[size_t(d.crop_plan)].K > CROP_KMAX) throw std::runtime_error("crops: crop scale");
            const PlanDev& np = plans_[size_t(d.canvas_plan)];
            const int k = crop_variant(np.K, np.fin, np.sw, i420);
            kn[size_t(i)] = k;
            ++first[k + 1];
            patch_w[k] = std::max(patch_w[k], d.pw);
            frame_w[k] = std::max(frame_w[k], d.new_w);
        }
        for (int k = 1; k <= CROP_VARIANTS; ++k) first[k] += first[k - 1];
        int at[CROP_VARIANTS];
        std::copy(first, first + CROP_VARIANTS, at);
        for (int i = 0; i < n; ++i) jd[at[kn[size_t(i)]]++] = all[size_t(i)];
        sync_plans();
        grow(jobs_dev_, jobs_bytes_, size_t(n) * sizeof(JobDev));
        CROP_CHECK(hipMemcpyAsync(jobs_dev_, jd, size_t(n) * sizeof(JobDev), hipMemcpyHostToDevice, s));
        hipError_t launched = hipSuccess;
        for (int k = 0; k < CROP_VARIANTS && launched == hipSuccess; ++k) {
            const int m = first[k + 1] - first[k];
            if (m == 0) continue;
            const CropSplit split = crop_split(n, k, frame_w[k]);
            const dim3 grid((CROP_H + split.band - 1) / split.band * split.chunks, m);
            const size_t lds = size_t(CROP_RING) * ring_width(patch_w[k], CROP_W / split.chunks) * 4;
            launch(std::make_integer_sequence<int, CROP_VARIANTS>(), i420, k, grid, lds, s,
                   static_cast<const JobDev*>(jobs_dev_) + first[k], out, split);
            launched = hipGetLastError();
        }
        const hipError_t done = hipStreamSynchronize(s);   // after a failed launch too: the next call reuses the job tables
        CROP_CHECK(launched);
        CROP_CHECK(done);
    }

private:
    typedef std::array<int, 6> Key;   // role, sw, sh, dw, dh, interpolation
    std::mutex mu_;
    int device_ = -1;
    std::map<Key, int> index_;
    std::vector<PlanDev> plans_;
    bool plans_dirty_ = false;
    void *plans_dev_ = nullptr, *jobs_dev_ = nullptr, *jobs_host_ = nullptr;
    size_t plans_bytes_ = 0, jobs_bytes_ = 0, jobs_host_bytes_ = 0;

    template <bool I420, int V>
    void launch_variant(dim3 grid, size_t lds, hipStream_t s, const JobDev* j, uint8_t* out, CropSplit split) {
        hipLaunchKernelGGL((crop_kernel<I420, V>), grid, dim3(CROP_THREADS), lds, s, j,
                           static_cast<const PlanDev*>(plans_dev_), out, split.band, split.chunks);
    }
    template <int... V>
    void launch(std::integer_sequence<int, V...>, bool i420, int v, dim3 grid, size_t lds, hipStream_t s, const JobDev* j,
                uint8_t* out, CropSplit split) {
        typedef void (CropEngine::*Go)(dim3, size_t, hipStream_t, const JobDev*, uint8_t*, CropSplit);
        static const Go go[2][CROP_VARIANTS] = {{&CropEngine::launch_variant<false, V>...},
                                                {&CropEngine::launch_variant<true, V>...}};
        (this->*go[i420][v])(grid, lds, s, j, out, split);
    }
    static void grow(void*& p, size_t& have, size_t need) {
        if (need <= have) return;
        if (p) CROP_CHECK(hipFree(p));
        p = nullptr;
        have = 0;
        CROP_CHECK(hipMalloc(&p, need));
        have = need;
    }
    static void grow_host(void*& p, size_t& have, size_t need) {   // pinned
        if (need <= have) return;
        if (p) CROP_CHECK(hipHostFree(p));
        p = nullptr;
        have = 0;
        CROP_CHECK(hipHostMalloc(&p, need, hipHostMallocDefault));
        have = need;
    }
    int plan_index(const Key& key) {
        const auto it = index_.find(key);
        if (it != index_.end()) return it->second;
        PlanHost h;
        if (!make_plan(key[1], key[2], key[3], key[4], key[5], h))
            throw std::runtime_error("crops: no resize plan for this geometry");
        // the plan's tables in one device allocation
        std::vector<uint32_t> words;
        const auto add = [&](const auto& v) {
            const size_t at = words.size();
            words.resize(at + v.size());
            std::memcpy(words.data() + at, v.data(), v.size() * 4);
            return at;
        };
        const size_t xoff = add(h.xoff), xw = add(h.xw), ysi = add(h.ysi), yw = add(h.yw);
        void* t = nullptr;
        CROP_CHECK(hipMalloc(&t, words.size() * 4));
        const hipError_t e = hipMemcpy(t, words.data(), words.size() * 4, hipMemcpyHostToDevice);
        if (e != hipSuccess) (void)hipFree(t);
        CROP_CHECK(e);
        const int* ti = static_cast<const int*>(t);
        const float* tf = static_cast<const float*>(t);
        PlanDev d;
        d.fin = h.fin; d.K = h.K; d.sw = h.sw; d.sh = h.sh; d.fscale = h.fscale;
        d.xoff = ti + xoff; d.xw = tf + xw; d.ysi = ti + ysi; d.yw = tf + yw;
        plans_.push_back(d);
        plans_dirty_ = true;
        return index_[key] = int(plans_.size() - 1);
    }
    void sync_plans() {
        if (!plans_dirty_) return;
        grow(plans_dev_, plans_bytes_, plans_.size() * sizeof(PlanDev));
        CROP_CHECK(hipMemcpy(plans_dev_, plans_.data(), plans_.size() * sizeof(PlanDev), hipMemcpyHostToDevice));
        plans_dirty_ = false;
    }
};

}  // namespace

void native_crops(const CropJob* jobs, int n, uint8_t* out, bool i420, hipStream_t s) {
    if (n <= 0) return;
    if (!jobs || !out || n > 65535) throw std::runtime_error("crops: null buffer or more than 65535 crops");
    CropEngine::get().run(jobs, n, out, s, i420);
}

}  // namespace shv
