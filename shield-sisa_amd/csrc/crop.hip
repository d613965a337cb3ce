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

// BT.601 limited-range coefficients of ffmpeg's yuv2rgb tables (contrast = saturation = 1 << 16, brightness 0),
// rounded to 16 bits as av_clip_int16((x + 2^15) >> 16): Y 76309 (= 65536 * 255 / 219) and the inverse-table
// entries 104597 (V->R), 132201 (U->B), -25675 (U->G), -53279 (V->G), each times 2^13; Y offset 16 << 19
struct Yuv {
    int y_coeff, vr, ub, ug, vg, y_off, uv_off;
};
__device__ __forceinline__ int sat16(int v) { return v < -32768 ? -32768 : (v > 32767 ? 32767 : v); }
__device__ __forceinline__ int mulhi16(int a, int b) { return (a * b) >> 16; }
__device__ __forceinline__ int sat8(int v) { return v < 0 ? 0 : (v > 255 ? 255 : v); }
__device__ __forceinline__ void yuv_px(const Yuv& k, int y, int u, int v, float (&o)[3]) {
    const int yp = int(short((y << 3) - k.y_off));
    const int up = sat16((u << 3) - k.uv_off), vp = sat16((v << 3) - k.uv_off);
    const int yy = mulhi16(yp, k.y_coeff);
    const int cg = sat16(mulhi16(up, k.ug) + mulhi16(vp, k.vg));
    o[0] = float(sat8(sat16(yy + mulhi16(vp, k.vr))));
    o[1] = float(sat8(sat16(yy + cg)));
    o[2] = float(sat8(sat16(yy + mulhi16(up, k.ub))));
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
    Yuv k;
    struct Row { GBytes y, u, v; };
    template <int K> struct Raw { unsigned y[load_words(K)], u[load_words(chroma_samples(K))], v[load_words(chroma_samples(K))]; };
    __device__ bool last(int y) const { return (y >> 1) == ((h + 1) >> 1) - 1; }
    __device__ Row row(int y) const {
        return {Y + (long long)y * ys, U + (long long)(y >> 1) * us, V + (long long)(y >> 1) * vs};
    }
    template <int K> __device__ void load(int x, const Row& q, Raw<K>& r) const {
        constexpr int C = chroma_samples(K);
        static_assert(load_words(C) == 1, "tap() picks the chroma samples out of one word");
        load_bytes<K>(q.y + unsigned(x), r.y);
        load_bytes<C>(q.u + (unsigned(x) >> 1), r.u);
        load_bytes<C>(q.v + (unsigned(x) >> 1), r.v);
    }
    template <int K> __device__ void tap(const Raw<K>& r, int x, int i, float (&o)[3]) const {
        const int sh = 8 * ((i + (x & 1)) >> 1);
        yuv_px(k, int(byte_of(r.y, i)), int((r.u[0] >> sh) & 255u), int((r.v[0] >> sh) & 255u), o);
    }
    __device__ void pixel(int x, const Row& q, float (&o)[3]) const {
        yuv_px(k, q.y[unsigned(x)], q.u[unsigned(x) >> 1], q.v[unsigned(x) >> 1], o);
    }
};
struct RingSrc {   // canvas rows in the LDS ring, one word (R, G, B) per pixel
    const unsigned* px;
    int pw;
    struct Row { const unsigned* p; };
    template <int K> struct Raw { unsigned px[K]; };
    __device__ Row row(int y) const { return {px + (y % CROP_RING) * pw}; }
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
#pragma unroll
        for (int k = 0; k < K; ++k) {
            float v[3];
            src.template tap<K>(raw[j], x0, k, v);
#pragma unroll
            for (int c = 0; c < 3; ++c) t[c] = k == 0 ? v[c] * w[k] : t[c] + v[c] * w[k];
        }
        col.add(j == 0, rows.b[j], t);
    }
    return col.finish(fscale);
}
// output pixel (x, y) of any plan, source pixel by source pixel, all inside the source
template <int FIN, class Src>
__device__ __forceinline__ unsigned resize_any_fin(const PlanDev& p, const Src& src, int x, int y) {
    const auto xw = (const AS_GLOBAL float*)p.xw;
    const int x0 = ((const AS_GLOBAL int*)p.xoff)[x];
    Column<FIN> col;
    for (int j = 0; j < p.K; ++j) {
        const typename Src::Row row = src.row(((const AS_CONST int*)p.ysi)[y * p.K + j]);
        float t[3] = {0.0f, 0.0f, 0.0f};
        for (int k = 0; k < p.K; ++k) {
            float v[3];
            src.pixel(min(x0 + k, p.sw - 1), row, v);
            const float a = xw[x * p.K + k];
#pragma unroll
            for (int c = 0; c < 3; ++c) t[c] = t[c] + v[c] * a;
        }
        col.add(j == 0, ((const AS_CONST float*)p.yw)[y * p.K + j], t);
    }
    return col.finish(p.fscale);
}
template <class Src> __device__ __forceinline__ unsigned resize_any(const PlanDev& p, const Src& src, int x, int y) {
    switch (p.fin) {
    case FIN_QUARTER: return resize_any_fin<FIN_QUARTER>(p, src, x, y);
    case FIN_LINEAR: return resize_any_fin<FIN_LINEAR>(p, src, x, y);
    default: return resize_any_fin<FIN_SCALE>(p, src, x, y);
    }
}

constexpr int CROP_THREADS = CROP_W, CROP_PASS = 1280 / CROP_THREADS;   // canvas columns per thread

// Canvas rows ya .. yb - 1 of the patch into the ring.  A thread keeps its (up to four) columns' taps for the whole band.
template <int K> struct Columns {
    int x0[CROP_PASS];
    float w[CROP_PASS][K ? K : 1];
};
template <int K, int FIN, class Src>
__device__ __forceinline__ void fill_rows(const JobDev& j, const PlanDev& p, const Src& src, const Columns<K>& cs, int ya,
                                          int yb, unsigned* ring) {
    const int passes = (j.pw + CROP_THREADS - 1) / CROP_THREADS, xa = j.px0 - j.left;
    const bool inside = xa >= 0 && xa + j.pw <= j.new_w;   // no letterbox bar left or right of the patch
    for (int r = ya; r < yb; ++r) {
        const int y = r + j.py0 - j.top;   // row of the resized frame; outside it the letterbox bars
        unsigned* row = ring + (r % CROP_RING) * j.pw;
        const bool bar = y < 0 || y >= j.new_h;
        if (K > 0 && !bar && !src.last(((const AS_CONST int*)p.ysi)[y * p.K + p.K - 1])) {
            if constexpr (K > 0) {
                const Rows<K, Src> rows(p, src, y);
#pragma unroll
                for (int q = 0; q < CROP_PASS; ++q) {
                    if (q >= passes) break;   // uniform; a column past the patch is computed (from its clamp) and dropped
                    const int px = threadIdx.x + CROP_THREADS * q;
                    unsigned v = resize_px<K, FIN>(rows, src, cs.x0[q], cs.w[q], p.fscale);
                    if (!inside) v = xa + px >= 0 && xa + px < j.new_w ? v : 0u;
                    if (px < j.pw) row[px] = v;
                }
            }
        } else {
            for (int px = threadIdx.x; px < j.pw; px += CROP_THREADS)
                row[px] = !bar && xa + px >= 0 && xa + px < j.new_w ? resize_any(p, src, xa + px, y) : 0u;
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
                                          int oy1, unsigned* ring, uint8_t* out) {
    Columns<K> cs;
#pragma unroll
    for (int q = 0; q < CROP_PASS; ++q) {
        const int px = threadIdx.x + CROP_THREADS * q, x = min(max(j.px0 + px - j.left, 0), j.new_w - 1);
        cs.x0[q] = ((const AS_GLOBAL int*)np.xoff)[x];
#pragma unroll
        for (int k = 0; k < K; ++k) cs.w[q][k] = ((const AS_GLOBAL float*)np.xw)[x * K + k];
    }
    const int ox = threadIdx.x;
    const int ox0 = ((const AS_GLOBAL int*)cp.xoff)[ox];
    float ow[CROP_KMAX];
#pragma unroll
    for (int k = 0; k < CROP_KMAX; ++k) ow[k] = k < cp.K ? ((const AS_GLOBAL float*)cp.xw)[ox * cp.K + k] : 0.0f;
    const auto ysi = (const AS_CONST int*)cp.ysi;
    const RingSrc rs{ring, j.pw};
    const bool words = (reinterpret_cast<uintptr_t>(out) & 3) == 0;
    uint8_t* d = out + 3 * CROP_W * oy0;
    int have = ysi[oy0 * cp.K];   // patch rows below this one are in the ring (or not needed)
    for (int oy = oy0; oy < oy1; ++oy, d += 3 * CROP_W) {
        const int need = ysi[oy * cp.K + cp.K - 1] + 1;
        fill_rows<K, FIN>(j, np, src, cs, have, need, ring);
        have = max(have, need);
        __syncthreads();
        const unsigned v = out_px_any(cp, rs, ox0, ow, oy);
        if (words) {
            const int i = ox & 3;
            const unsigned w = quad_word(v, i);
            if (i < 3) *reinterpret_cast<unsigned*>(d + 3 * (ox - i) + 4 * i) = w;
        } else {
            d[3 * ox] = uint8_t(v);
            d[3 * ox + 1] = uint8_t(v >> 8);
            d[3 * ox + 2] = uint8_t(v >> 16);
        }
        __syncthreads();   // the next rows go into slots that this row's threads may still read
    }
}

// Workgroup (band of output rows, crop) of five waves: per output row the canvas rows it adds (each thread its columns,
// so a wave reads neighbouring pixels), then one output pixel per thread.  Reads the native pixels under a crop once (a
// row or two more per band) and writes the crop; bound by the instructions of the row pass: a conversion, a product and
// a sum per byte and tap.
// Kernel time of 640 crops of 1920 x 1080 RGB frames 1.24 ms, of 80 crops of 1280 x 720 I420 frames 156 us; the calls 6.44 ->
// 1.83 ms and 414 -> 237 us (two kernels, canvas patches through HBM, tap loops over byte loads before).
template <bool I420, int V>
__global__ void __launch_bounds__(CROP_THREADS)
crop_kernel(const JobDev* __restrict__ jobs, const PlanDev* __restrict__ plans, uint8_t* __restrict__ out, Yuv yuv,
            int band) {
    extern __shared__ __attribute__((aligned(16))) unsigned ring[];
    constexpr int K = kVariants[V].K, FIN = kVariants[V].fin;
    const JobDev j = jobs[blockIdx.y];
    const int oy0 = blockIdx.x * band, oy1 = min(CROP_H, oy0 + band);
    const PlanDev cp = plans[j.crop_plan], np = plans[j.canvas_plan];
    uint8_t* d = out + (long long)j.index * (CROP_W * CROP_H * 3);
    if constexpr (I420) {
        const I420Src src{global_bytes(j.frame), global_bytes(j.u), global_bytes(j.v), j.stride, j.u_stride, j.v_stride,
                          np.sh, yuv};
        crop_band<K, FIN>(j, np, cp, src, oy0, oy1, ring, d);
    } else {
        const RgbSrc src{global_bytes(j.frame), j.stride, np.sh};
        crop_band<K, FIN>(j, np, cp, src, oy0, oy1, ring, d);
    }
}

// 16-bit rounding of a 2^16-scaled coefficient with saturation (ffmpeg's round + av_clip_int16)
int round_to_16(long long f) {
    int r = int((f + (1 << 15)) >> 16);
    if (r < -32768) r = -32768;
    if (r > 32767) r = 32767;
    return r;
}
Yuv yuv_coeffs() {
    const long long cy = (65536LL * 255) / 219;   // contrast = saturation = 1 << 16 leave the table entries unscaled
    Yuv k;
    k.y_coeff = round_to_16(cy * (1 << 13));
    k.vr = round_to_16(104597LL * (1 << 13));
    k.ub = round_to_16(132201LL * (1 << 13));
    k.ug = round_to_16(-25675LL * (1 << 13));
    k.vg = round_to_16(-53279LL * (1 << 13));
    k.y_off = round_to_16((16LL << 16) * (1 << 3));
    k.uv_off = 0x0400;
    return k;
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
        int first[CROP_VARIANTS + 1] = {}, width[CROP_VARIANTS] = {};   // crops of each variant, widest patch
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
            width[k] = std::max(width[k], d.pw);
        }
        for (int k = 1; k <= CROP_VARIANTS; ++k) first[k] += first[k - 1];
        int at[CROP_VARIANTS];
        std::copy(first, first + CROP_VARIANTS, at);
        for (int i = 0; i < n; ++i) jd[at[kn[size_t(i)]]++] = all[size_t(i)];
        sync_plans();
        grow(jobs_dev_, jobs_bytes_, size_t(n) * sizeof(JobDev));
        CROP_CHECK(hipMemcpyAsync(jobs_dev_, jd, size_t(n) * sizeof(JobDev), hipMemcpyHostToDevice, s));
        // bands per crop: enough workgroups for a few crops, 15 output rows each for many (a band recomputes a canvas
        // row or two)
        const int bands = std::max(12, std::min(60, (6144 + n - 1) / n)), band = (CROP_H + bands - 1) / bands;
        static const Yuv yuv = yuv_coeffs();
        for (int k = 0; k < CROP_VARIANTS; ++k) {
            const int m = first[k + 1] - first[k];
            if (m == 0) continue;
            const dim3 grid((CROP_H + band - 1) / band, m);
            const size_t lds = size_t(CROP_RING) * width[k] * 4;
            launch(std::make_integer_sequence<int, CROP_VARIANTS>(), i420, k, grid, lds, s, static_cast<const JobDev*>(jobs_dev_) + first[k], out, yuv, band);
            CROP_CHECK(hipGetLastError());
        }
        CROP_CHECK(hipStreamSynchronize(s));   // the job table is reused by the next call
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
    void launch_variant(dim3 grid, size_t lds, hipStream_t s, const JobDev* j, uint8_t* out, const Yuv& yuv, int band) {
        hipLaunchKernelGGL((crop_kernel<I420, V>), grid, dim3(CROP_THREADS), lds, s, j,
                           static_cast<const PlanDev*>(plans_dev_), out, yuv, band);
    }
    template <int... V>
    void launch(std::integer_sequence<int, V...>, bool i420, int v, dim3 grid, size_t lds, hipStream_t s, const JobDev* j,
                uint8_t* out, const Yuv& yuv, int band) {
        typedef void (CropEngine::*Go)(dim3, size_t, hipStream_t, const JobDev*, uint8_t*, const Yuv&, int);
        static const Go go[2][CROP_VARIANTS] = {{&CropEngine::launch_variant<false, V>...},
                                                {&CropEngine::launch_variant<true, V>...}};
        (this->*go[i420][v])(grid, lds, s, j, out, yuv, band);
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
