// Expand + depthwise of an inverted-residual block in one kernel: X [n][H][W][K] -> (1x1 convolution, bias, activation)
// -> (depthwise KS x KS, strides SY / SX) -> D [n][Ho][Wo][C].  The expanded map E, 2 to 4 times the block's other maps
// together, stays in LDS.  Two users: the exact tier's blocks 2-15 (activations fp32, the reference CPU engine's
// operation order: engine/model/isa_impl.hpp:188-317, 603-643) and the SHIELD-A frontend's eight blocks in every tier
// (engine/audio/frontend.cpp:193-204).
//
// A workgroup of eight waves owns a band of BR output rows (all columns) of NI images.  It reads the band's input pixels
// once, as the MFMA A fragments of 16-pixel tiles (tile t to wave t % 8) that stay in registers, and then walks the
// expanded channels 16 at a time: each wave multiplies its tiles with the chunk's weights, writes the activated
// 16 x 16 results to the LDS tile [row][column][16 + pad] (rows and columns outside the map zero, as the layer pads E),
// and after a barrier each thread takes one channel of R consecutive output rows at a time, loading its window once.
// Per output the operations and their order are those of the GEMM's and the depthwise layer's kernels (fp32: bitwise
// theirs; SHIELD-A: sum of products over (kf, kt), BatchNorm, SiLU as silu_near()).  Few images: the chunks are dealt
// over blockIdx.y too.
//
// Bound (MFMA / VALU busy by counters): SHIELD-A's early blocks by vector instructions, SiLU and depthwise (A0 6 / 96%, A1 7
// / 68%), B2-B4 by them and memory (17-30 / 30-36% at 1.8-2.7 TB/s), the late blocks of both by a workgroup's waits between
// its barriers, with one and a half waves a SIMD (B13 23 / 19%, B14 14 / 18%, A5 6 / 27%, A7 6 / 22%).  So SiLU is the
// 16-instruction form, and the next chunk's expand weights are read before the depthwise's stores (a load behind a store
// waits for it).  Against the expand GEMM and the depthwise kernel apart, which wrote and read E: 32 clips in fp32 11.30 ->
// 9.36 ms, one clip 1214 -> 1142 us; 128 SHIELD-A windows fp16 13.9 -> 11.5 ms, 5 windows fp32 967 -> 939 us.  SHIELD-A's
// first block also computes its input, the stem, from the log-mel tile in LDS, once per band in the fragments' own layout: a stem kernel
// wrote 163 MB per 16 windows in 113 us (each thread loaded its 72 weights) and the block took 105 us; together 125 us,
// 128 windows fp16 11.5 -> 10.6 ms, 5 windows fp32 939 -> 907 us.
#include "dev_common.hpp"
#include "gemm_f32.hpp"
#include "kernels.hpp"
#include "mfma.hpp"

#include <algorithm>
#include <stdexcept>
#include <string>
#include <type_traits>

namespace shv {
namespace {

inline unsigned int cdiv(long long a, long long b) { return (unsigned int)((a + b - 1) / b); }

constexpr int ED_WAVES = 8, ED_THREADS = 64 * ED_WAVES;
constexpr int ED_CS = 16 + 4;   // LDS floats per pixel: the four pixel rows of an accumulator write fall on distinct banks

// Geometry of one block.  MODE: activation and depthwise arithmetic.
enum { ED_RELU = 0, ED_HS = 1, ED_AUDIO = 2, ED_STEM = 3 };   // ED_STEM: ED_AUDIO, X computed from the log-mel image
template <int H_, int W_, int K_, int C_, int KS_, int SY_, int SX_, int MODE_, int BR_, int NI_, int R_, int WGS_ = 1>
struct EdShape {
    static constexpr int H = H_, W = W_, K = K_, C = C_, KS = KS_, SY = SY_, SX = SX_, MODE = MODE_, BR = BR_, NI = NI_, R = R_,
                         WGS = WGS_;   // workgroups a CU is to hold (registers)
    static constexpr int P = (KS - 1) / 2, Ho = (H - 1) / SY + 1, Wo = (W - 1) / SX + 1;
    static constexpr int RI = (BR - 1) * SY + KS, WP = W + 2 * P;            // LDS rows per image, pixels per LDS row
    static constexpr int RV = RI < H ? RI : H;                               // most input rows of a band inside the map
    static constexpr int MT = (NI * RV * W + 16 * ED_WAVES - 1) / (16 * ED_WAVES);   // tiles per wave
    static constexpr int CHUNKS = (C + 15) / 16, BANDS = (Ho + BR - 1) / BR;
    static constexpr int GROUPS = (BR + R - 1) / R, UNITS = NI * GROUPS * Wo, WR = (R - 1) * SY + KS;
    // window rows of the last group reach past the tile when R does not divide BR: the LDS tile has them
    static constexpr int RL = (GROUPS * R - 1) * SY + KS, E_LDS = NI * RL * WP * ED_CS;
    // ED_STEM: after E the band's log-mel rows and columns with a border of one, then the stem's weights [9][32], scale, shift
    static constexpr bool AUDIO = MODE >= ED_AUDIO, STEM = MODE == ED_STEM;
    static constexpr int MELW = W + 2, MEL = ((RV + 2) * MELW + 3) / 4 * 4, LDS = E_LDS + (STEM ? MEL + 11 * 32 : 0);
    static_assert(NI == 1 || BR >= Ho, "several images: whole maps");
    static_assert(!STEM || (K == 32 && NI == 1), "the stem has 32 channels");
};

// one 16 x 16 x K product in the tier's arithmetic; fragments as the GEMM kernels'

template <typename T, int K> struct EdMma {   // half types: K steps of 32, split products in order
    static constexpr int P = Split<T>::P, NS = (K + 31) / 32;
    typedef typename Split<T>::V8 V8;
    struct A { V8 v[NS][P]; };
    struct B { V8 v[NS][P]; };
    template <class X4> static __device__ __forceinline__ void load_a(A& a, X4&& x4, int g) {   // x4(k): X[k .. k + 3]
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int k = 32 * s + 8 * g;
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = 0.0f;
            if (K % 32 == 0 || k < K) {
                const f32x4 lo = x4(k), hi = x4(k + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[e] = lo[e];
                    x[4 + e] = hi[e];
                }
            }
            split8<T>(x, a.v[s]);
        }
    }
    static __device__ __forceinline__ void load_b(B& b, const void* w, long long wstride, int n, int g) {
        const T* row = static_cast<const T*>(w) + (long long)n * K;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int k = 32 * s + 8 * g;
#pragma unroll
            for (int q = 0; q < P; ++q) {
                V8 z = {};
                if (K % 32 == 0 || k < K) z = load_part8<T>(row + q * wstride + k);
                b.v[s][q] = z;
            }
        }
    }
    static __device__ __forceinline__ void prepare_b(B&) {}
    static __device__ __forceinline__ f32x4 mul(const A& a, const B& b) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < NS; ++s) acc = mfma_split<T>(a.v[s], b.v[s], acc);
        return acc;
    }
};
template <int K> struct EdMma<float, K> {   // the reference's K blocks of 64 (gemm_f32.hip)
    static constexpr int NC = (K + 15) / 16;
    struct A { float v[NC][4]; };
    struct B { f32x4 v[NC]; };
    template <class X4> static __device__ __forceinline__ void load_a(A& a, X4&& x4, int g) {
        f32x4 x[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) x[c] = x4(min(16 * c + 4 * g, K - 4));
#pragma unroll
        for (int c = 0; c < NC; ++c) transpose4(x[c], a.v[c]);
    }
    static __device__ __forceinline__ void load_b(B& b, const void* w, long long, int n, int g) {
        const float* row = static_cast<const float*>(w) + (long long)n * K;
#pragma unroll
        for (int c = 0; c < NC; ++c) b.v[c] = ld4(row + min(16 * c + 4 * g, K - 4));
    }
    static __device__ __forceinline__ void prepare_b(B& b) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            float t[4];
            transpose4(b.v[c], t);
            b.v[c] = f32x4{t[0], t[1], t[2], t[3]};
        }
    }
    static __device__ __forceinline__ f32x4 mul(const A& a, const B& b) {
        f32x4 tot = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k0 = 0; k0 < K; k0 += 64) {
            f32x4 blk = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = k0; k < K && k < k0 + 64; k += 4) blk = mfma4(a.v[k / 16][(k / 4) % 4], b.v[k / 16][(k / 4) % 4], blk);
            tot = k0 == 0 ? blk : tot + blk;
        }
        return tot;
    }
};

// LDS accesses of the workgroup done; loads and stores to memory stay in flight
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <typename T, class S>
__global__ void __launch_bounds__(ED_THREADS, (std::is_same<T, bf16>::value ? 1 : S::WGS) * ED_WAVES / 4) expdw_kernel(ExpDwArgs p) {
    typedef EdMma<T, S::K> M;
    extern __shared__ __attribute__((aligned(16))) float E[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, r = lane & 15;
    const int img0 = (blockIdx.x / S::BANDS) * S::NI, oy0 = (blockIdx.x % S::BANDS) * S::BR;
    const int imgs = min(S::NI, p.n - img0);
    const int iy0 = oy0 * S::SY - S::P;                                   // map row of LDS row 0
    const int va = max(iy0, 0), vb = min(S::H, iy0 + S::RI);              // rows inside the map
    const int m_end = imgs * (vb - va) * S::W;                            // pixels (several images: whole maps)
    const int per = (S::CHUNKS + gridDim.y - 1) / gridDim.y;
    const int ch0 = blockIdx.y * per, ch1 = min(S::CHUNKS, ch0 + per);
    if (ch0 >= ch1) return;   // uniform over the workgroup

    typename M::A a[S::MT];   // tiles past the band read its last pixel and are not used
    if constexpr (S::STEM) {
        float *mel = E + S::E_LDS, *sw = mel + S::MEL;
        const float* src = p.X + (long long)img0 * (S::H * S::W);
        for (int i = tid; i < (vb - va + 2) * S::MELW; i += ED_THREADS) {
            const int y = va - 1 + i / S::MELW, x = i % S::MELW - 1;
            mel[i] = y >= 0 && y < S::H && x >= 0 && x < S::W ? src[y * S::W + x] : 0.0f;
        }
        for (int i = tid; i < 11 * 32; i += ED_THREADS)
            sw[i] = i < 288 ? p.stem_w[(i & 31) * 9 + (i >> 5)] : i < 320 ? p.stem_scale[i - 288] : p.stem_shift[i - 320];
        lds_barrier();
#pragma unroll
        for (int t = 0; t < S::MT; ++t) {
            const int m = min((wave + ED_WAVES * t) * 16 + r, m_end - 1), row = m / S::W, col = m - row * S::W;
            float tap[9];   // (kf, kt)
#pragma unroll
            for (int q = 0; q < 9; ++q) tap[q] = mel[(row + q % 3) * S::MELW + col + q / 3];
            M::load_a(a[t], [&](int k) {
                f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int q = 0; q < 9; ++q) {
                    const f32x4 w = ld4(sw + q * 32 + k);
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[e] = __builtin_fmaf(tap[q], w[e], s[e]);
                }
                const f32x4 sc = ld4(sw + 288 + k), sh = ld4(sw + 320 + k);
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] = silu_near(s[e] * sc[e] + sh[e]);
                return s;
            }, g);
        }
    } else {
        const float* x0 = p.X + ((long long)img0 * S::H + va) * (S::W * S::K);
#pragma unroll
        for (int t = 0; t < S::MT; ++t) {
            const float* row = x0 + (long long)min((wave + ED_WAVES * t) * 16 + r, m_end - 1) * S::K;
            M::load_a(a[t], [&](int k) { return ld4(row + k); }, g);
        }
    }
    typename M::B b;
    const auto fetch = [&](int ch, float& eb) {   // a chunk's expand weights and bias
        const int n = min(ch * 16 + r, S::C - 1);
        M::load_b(b, p.W, p.wstride, n, g);
        eb = p.bexp[n];
    };
    float eb_next;
    fetch(ch0, eb_next);
    for (int i = tid; i < S::E_LDS / 4; i += ED_THREADS) reinterpret_cast<f32x4*>(E)[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // LDS position of the lane's first pixel of each tile (of each pixel where a row is no multiple of four)
    constexpr int PI = S::W % 4 == 0 ? 1 : 4;
    int eo[S::MT][PI];
#pragma unroll
    for (int t = 0; t < S::MT; ++t)
#pragma unroll
        for (int i = 0; i < PI; ++i) {
            const int m = (wave + ED_WAVES * t) * 16 + 4 * g + i;
            const int row = m / S::W, col = m - row * S::W, img = S::NI == 1 ? 0 : row / S::H;
            const int lr = S::NI == 1 ? row + va - iy0 : img * S::RL + row - img * S::H + S::P;
            eo[t][i] = m < m_end ? (lr * S::WP + S::P + col) * ED_CS + r : -1;
        }
    // depthwise: channel of the chunk, then this thread's units (image, group of R output rows, column): LDS position of
    // the window, offset of the first output, rows to store
    constexpr int UP = (S::UNITS + ED_THREADS / 16 - 1) / (ED_THREADS / 16);
    const int dc = tid & 15;
    int uo[UP], od[UP], rows[UP];
#pragma unroll
    for (int k = 0; k < UP; ++k) {
        const int u = min((tid >> 4) + ED_THREADS / 16 * k, S::UNITS - 1);
        const int ox = u % S::Wo, q = u / S::Wo, grp = q % S::GROUPS, img = q / S::GROUPS;
        uo[k] = ((img * S::RL + grp * S::R * S::SY) * S::WP + ox * S::SX) * ED_CS + dc;
        od[k] = ((img * S::Ho + grp * S::R) * S::Wo + ox) * S::C + dc;
        rows[k] = img < imgs && (tid >> 4) + ED_THREADS / 16 * k < S::UNITS
                      ? min(S::R, min(S::BR, S::Ho - oy0) - grp * S::R) : 0;
    }
    float* d0 = p.D + ((long long)img0 * S::Ho + oy0) * S::Wo * S::C;
    lds_barrier();

    for (int ch = ch0; ch < ch1; ++ch) {
        const float eb = eb_next;
        M::prepare_b(b);
        const int cc = min(ch * 16 + dc, S::C - 1);
        float w[S::KS * S::KS];
#pragma unroll
        for (int q = 0; q < S::KS * S::KS; ++q) w[q] = p.wdw[q * S::C + cc];
        const float db = p.bdw[cc], ds = S::AUDIO ? p.sdw[cc] : 1.0f;
#pragma unroll
        for (int t = 0; t < S::MT; ++t) {
            if ((wave + ED_WAVES * t) * 16 >= m_end) break;   // uniform over the wave
            const f32x4 acc = M::mul(a[t], b);
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = (std::is_same<T, float>::value ? acc[i] : acc[i] * p.wscale) + eb;
            if constexpr (S::MODE == ED_RELU) apply_act4<ACT_RELU>(v);
            else if constexpr (S::MODE == ED_HS) apply_act4<ACT_HS>(v);
            else {
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = silu_near(v[i]);
            }
            if constexpr (PI == 1) {   // the lane's four pixels share a row, and m_end % 4 == 0
                if (eo[t][0] >= 0) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) E[eo[t][0] + i * ED_CS] = v[i];
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (eo[t][i] >= 0) E[eo[t][i]] = v[i];
            }
        }
        if (ch + 1 < ch1) fetch(ch + 1, eb_next);
        lds_barrier();
        float* d = d0 + ch * 16;
        const bool live = ch * 16 + dc < S::C;
#pragma unroll
        for (int k = 0; k < UP; ++k) {
            const float* e = E + uo[k];
            float win[S::WR][S::KS];
#pragma unroll
            for (int y = 0; y < S::WR; ++y)
#pragma unroll
                for (int x = 0; x < S::KS; ++x) win[y][x] = e[(y * S::WP + x) * ED_CS];
#pragma unroll
            for (int o = 0; o < S::R; ++o) {
                float s = 0.0f, v;
                if constexpr (S::AUDIO) {   // columns (frequency) outer, rows (time) inner; product, then sum
#pragma unroll
                    for (int x = 0; x < S::KS; ++x)
#pragma unroll
                        for (int y = 0; y < S::KS; ++y) s = s + win[o * S::SY + y][x] * w[x * S::KS + y];
                    v = silu_near(s * ds + db);
                } else {
#pragma unroll
                    for (int y = 0; y < S::KS; ++y)
#pragma unroll
                        for (int x = 0; x < S::KS; ++x) s = __builtin_fmaf(win[o * S::SY + y][x], w[y * S::KS + x], s);
                    v = apply_act(s + db, S::MODE == ED_HS ? ACT_HS : ACT_RELU);
                }
                if (live && o < rows[k]) d[od[k] + o * (S::Wo * S::C)] = v;
            }
        }
        lds_barrier();   // the next chunk overwrites E
    }
}

template <typename T, class S> void launch_shape(const ExpDwArgs& p, hipStream_t s) {
    const long long wgs = (long long)cdiv(p.n, S::NI) * S::BANDS;
    if (wgs >= (1ll << 31)) throw std::runtime_error("expdw: grid too large");
    constexpr size_t lds = size_t(S::LDS) * 4;
    static_assert(lds <= 160 * 1024, "LDS tile");
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(expdw_kernel<T, S>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
        if (e != hipSuccess) throw std::runtime_error(std::string("expdw: ") + hipGetErrorString(e));
    }
    // few bands: the chunks dealt over as many workgroups as the device holds at once (each loads the band's X again)
    static const int per_cu = [] {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void*>(expdw_kernel<T, S>), ED_THREADS,
                                                         lds) != hipSuccess)
            n = 1;
        return std::max(1, n);
    }();
    const int split = int(std::max(1ll, std::min((long long)S::CHUNKS, 256ll * per_cu / wgs)));
    hipLaunchKernelGGL((expdw_kernel<T, S>), dim3((unsigned)wgs, split), dim3(ED_THREADS), lds, s, p);
}

// Bands: as few input rows computed twice as two workgroups a CU (LDS 80 KB each, 128 registers a lane) allow.  Where the
// A fragments alone pass that (B5, B13, B14, A5, A7) the band is larger and one workgroup holds the CU: A5 in bands of 4
// rows and two workgroups took 87 us to 82.  A1 and A2 differ by type: in the half types, whose split A fragments are
// larger, 10 rows left one workgroup a CU (A1 124 us at 16 windows, 7 rows 87); in fp32 they hold two (38 us at 5
// windows, 7 rows 49).
//                       H    W   K    C  KS SY SX  MODE    BR NI R
typedef EdShape<90, 160, 16, 64, 3, 2, 2, ED_RELU, 2, 1, 2> B2;
typedef EdShape<45, 80, 24, 72, 3, 1, 1, ED_RELU, 9, 1, 3> B3;
typedef EdShape<45, 80, 24, 72, 5, 2, 2, ED_RELU, 4, 1, 1, 2> B4;
typedef EdShape<23, 40, 40, 120, 5, 1, 1, ED_RELU, 12, 1, 4> B5;
typedef EdShape<23, 40, 40, 240, 3, 2, 2, ED_HS, 6, 1, 2> B7;
typedef EdShape<12, 20, 80, 200, 3, 1, 1, ED_HS, 12, 1, 4> B8;
typedef EdShape<12, 20, 80, 184, 3, 1, 1, ED_HS, 12, 1, 4> B9;
typedef EdShape<12, 20, 80, 480, 3, 1, 1, ED_HS, 12, 1, 4> B11;
typedef EdShape<12, 20, 112, 672, 3, 1, 1, ED_HS, 12, 1, 2, 2> B12;
typedef EdShape<12, 20, 112, 672, 5, 2, 2, ED_HS, 6, 1, 2> B13;
typedef EdShape<6, 10, 160, 960, 5, 1, 1, ED_HS, 6, 2, 2> B14;
typedef EdShape<997, 80, 32, 64, 3, 2, 2, ED_STEM, 4, 1, 2, 2> A0;
typedef EdShape<499, 40, 48, 96, 3, 1, 1, ED_AUDIO, 10, 1, 5, 2> A1;   // fp32
typedef EdShape<499, 40, 48, 96, 3, 1, 1, ED_AUDIO, 7, 1, 2, 2> A1H;   // half types
typedef EdShape<499, 40, 48, 96, 3, 2, 2, ED_AUDIO, 5, 1, 5, 2> A2;
typedef EdShape<499, 40, 48, 96, 3, 2, 2, ED_AUDIO, 4, 1, 2, 2> A2H;
typedef EdShape<250, 20, 96, 192, 3, 1, 1, ED_AUDIO, 10, 1, 2, 2> A3;
typedef EdShape<250, 20, 96, 192, 3, 2, 1, ED_AUDIO, 5, 1, 2, 2> A4;
typedef EdShape<125, 20, 160, 320, 3, 1, 1, ED_AUDIO, 10, 1, 5> A5;
typedef EdShape<125, 20, 192, 384, 3, 1, 1, ED_AUDIO, 10, 1, 5> A7;

void check(const ExpDwArgs& p) {
    const auto al16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    if (p.n < 1 || !p.X || !p.D || !p.W || !al16(p.X) || !al16(p.W)) throw std::runtime_error("expdw: bad operands");
}
}  // namespace

void launch_expdw_f32(int block, const ExpDwArgs& p, hipStream_t s) {
    check(p);
    switch (block) {
    case 2: launch_shape<float, B2>(p, s); return;
    case 3: launch_shape<float, B3>(p, s); return;
    case 4: launch_shape<float, B4>(p, s); return;
    case 5: case 6: launch_shape<float, B5>(p, s); return;
    case 7: launch_shape<float, B7>(p, s); return;
    case 8: launch_shape<float, B8>(p, s); return;
    case 9: case 10: launch_shape<float, B9>(p, s); return;
    case 11: launch_shape<float, B11>(p, s); return;
    case 12: launch_shape<float, B12>(p, s); return;
    case 13: launch_shape<float, B13>(p, s); return;
    case 14: case 15: launch_shape<float, B14>(p, s); return;
    }
    throw std::runtime_error("expdw: no such block");
}
template <typename T> void launch_audio_expdw(int block, const ExpDwArgs& p, hipStream_t s) {
    check(p);
    if (block == 0 && (!p.stem_w || !p.stem_scale || !p.stem_shift)) throw std::runtime_error("expdw: bad operands");
    switch (block) {
    case 0: launch_shape<T, A0>(p, s); return;
    case 1: launch_shape<T, std::conditional_t<std::is_same<T, float>::value, A1, A1H>>(p, s); return;
    case 2: launch_shape<T, std::conditional_t<std::is_same<T, float>::value, A2, A2H>>(p, s); return;
    case 3: launch_shape<T, A3>(p, s); return;
    case 4: launch_shape<T, A4>(p, s); return;
    case 5: case 6: launch_shape<T, A5>(p, s); return;
    case 7: launch_shape<T, A7>(p, s); return;
    }
    throw std::runtime_error("expdw: no such block");
}
template void launch_audio_expdw<float>(int, const ExpDwArgs&, hipStream_t);
template void launch_audio_expdw<f16>(int, const ExpDwArgs&, hipStream_t);
template void launch_audio_expdw<bf16>(int, const ExpDwArgs&, hipStream_t);

}  // namespace shv
