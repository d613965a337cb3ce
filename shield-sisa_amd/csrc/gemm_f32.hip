// Exact-tier GEMMs on the fp32 matrix cores in the reference CPU engine's operation order.
//
// v_mfma_f32_16x16x4_f32 is, per output, four fused multiply-adds in increasing k onto its accumulator, each rounded
// to nearest even (checked bit for bit against the fma chain on the device: normal, subnormal and zero operands,
// 40-binade spreads, infinities and NaN).  A K block of 64 is therefore 16 MFMAs chained from +0, and the block sums
// added left to right give exactly the per-element sequence of the reference (engine/model/isa_impl.hpp:188-317) and
// of the VALU kernels in gemm.hip: bitwise the same results from twice their arithmetic rate (the matrix cores'
// 157 TFLOP/s against 79 of unpacked fp32 fmas).
#include "dev_common.hpp"
#include "gemm_f32.hpp"
#include "kernels.hpp"

#include <stdexcept>
#include <string>
#include <type_traits>

namespace shv {
namespace {

inline unsigned int cdiv(long long a, long long b) { return (unsigned int)((a + b - 1) / b); }

constexpr int KBLK = 64;   // the reference's K block
constexpr int XCDS = 8;

// the k steps of a 16-k chunk of which `left` (a positive multiple of 4) remain: exactly K's, since a zero product
// past K would turn a chain's -0 into +0
template <class Step> __device__ __forceinline__ void steps(int left, Step step) {
    if (left >= 16) {
        step(0); step(1); step(2); step(3);
        return;
    }
    step(0);
    if (left > 4) step(1);
    if (left > 8) step(2);
}
// epi_value's operations on the J x 4 outputs of one 16-row strip, the flags tested once per strip instead of once per
// output (vector instructions are what the matrix cores wait for here)
template <int J> __device__ __forceinline__ void activate(float (&v)[J][4], int act) {
    switch (act) {
    case ACT_RELU:
#pragma unroll
        for (int j = 0; j < J; ++j) apply_act4<ACT_RELU>(v[j]);
        return;
    case ACT_HS:
#pragma unroll
        for (int j = 0; j < J; ++j) apply_act4<ACT_HS>(v[j]);
        return;
    case ACT_HSIG:
#pragma unroll
        for (int j = 0; j < J; ++j) apply_act4<ACT_HSIG>(v[j]);
        return;
    case ACT_SILU:
#pragma unroll
        for (int j = 0; j < J; ++j) apply_act4<ACT_SILU>(v[j]);
        return;
    }
}
// Outputs of one 16-row strip of J column tiles: sum[j][i] at row m0 + 4 g + i, column n0 + 16 j + r.  Every bias and
// residual operand is loaded (at clamped, valid addresses) before the first store (see epi_block).
// swiglu 1: columns (2 q, 2 q + 1) = (gate, up) of output q; 2: tiles (2 q, 2 q + 1) = 16 gates, 16 ups.
template <int J>
__device__ __forceinline__ void store_strip(const GemmArgs& p, int swiglu, long long m0, int n0, int g, int r,
                                            const f32x4 (&sum)[J]) {
    if (swiglu) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const long long m = m0 + 4 * g + i;
            if (swiglu == 1) {
#pragma unroll
                for (int j = 0; j < J; ++j) {
                    const float v = sum[j][i], up = __shfl_xor(v, 1);
                    const int n = n0 + 16 * j + r;
                    if (m < p.M && !(r & 1) && n + 1 < p.N) p.C[m * p.ldc + (n >> 1)] = silu(v) * up;
                }
            } else if (m < p.M) {
#pragma unroll
                for (int j = 0; j + 1 < J; j += 2) {
                    const int panel = n0 / 16 + j;
                    if ((panel + 1) * 16 <= p.N) p.C[m * p.ldc + (panel / 2) * 16 + r] = silu(sum[j][i]) * sum[j + 1][i];
                }
            }
        }
        return;
    }
    if (m0 >= p.M) return;
    const int rows = int(min(16ll, p.M - m0));   // of the strip; uniform, as the column count
    const bool whole = rows == 16 && n0 + 16 * J <= p.N;
    float v[J][4], res[J][4];
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[j][i] = sum[j][i];
    if (p.res) {
        const float* R = p.R + m0 * p.ldr;
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) res[j][i] = R[min(4 * g + i, rows - 1) * (int)p.ldr + min(n0 + 16 * j + r, p.N - 1)];
    }
    if (p.bias) {
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const float b = p.bias[min(n0 + 16 * j + r, p.N - 1)];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[j][i] = v[j][i] + b;
        }
    }
    activate(v, p.act);
    if (p.res) {
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                v[j][i] = p.res == 3 ? res[j][i] + 0.7071067811865475244f * v[j][i]
                                     : p.res == 2 ? res[j][i] + v[j][i] / 1.41421356237309515f : res[j][i] + v[j][i];
    }
    float* C = p.C + m0 * p.ldc + n0;
    const int o = 4 * g * (int)p.ldc + r;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < J; ++j)
            if (whole || (4 * g + i < rows && n0 + 16 * j + r < p.N)) C[o + i * (int)p.ldc + 16 * j] = v[j][i];
}

// ------------------------------------------------------------------------------------------------ tiled
// A workgroup of four waves owns 64 rows x 16 WN columns, a wave 16 rows of it.  K is staged through LDS 32 at
// a time (two 16-k chunks, each [row][16] so that a fragment read of 64 lanes is 1 KB in a row and the 8-lane row
// loads write whole rows), the next 32 in registers meanwhile; the second buffer makes it one barrier per stage.
// Bound by the matrix cores where K is long (an MFMA takes 32 cycles, its operands 1/2 float4 of LDS): 69% busy in the
// 41,088-row sequence GEMMs, the LDS 36% (half of it bank conflicts), 2.8 waves a SIMD; 28-51% in the
// encoder's layers, at 4.1 (72 -> 24) to 0.8 TB/s (160 -> 960).
constexpr int TSTAGE = 32;
template <int WN, bool SCALE>
__global__ void __launch_bounds__(256, 3) gemm_f32_tile_kernel(GemmArgs p, int swiglu, int mblocks, int nblocks) {
    constexpr int BM = 64, BN = 16 * WN, GM = 8;
    constexpr int ACH = BM * 16 + 8, WCH = BN * 16 + 8;   // floats per chunk; the pad keeps the two chunks' banks apart
    constexpr int APT = BM / 32, WPT = (BN + 31) / 32;      // float4s per thread and stage
    __shared__ __attribute__((aligned(16))) float As[2][2 * ACH];
    __shared__ __attribute__((aligned(16))) float Ws[2][2 * WCH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, r = lane & 15;
    // workgroups go round robin over the XCDs; XCD x takes M blocks 8 i + x, in groups of GM of them column block by
    // column block, so that a group's A and the W blocks stay in its L2
    const int xcd = blockIdx.x % XCDS, slot = blockIdx.x / XCDS;
    const int mloc = (mblocks + XCDS - 1) / XCDS;
    const int grp = slot / (GM * nblocks), within = slot % (GM * nblocks);
    const int gsize = min(GM, mloc - grp * GM);
    const int mb = (grp * GM + within % gsize) * XCDS + xcd, nb = within / gsize;
    if (mb >= mblocks) return;   // uniform over the workgroup
    const long long m0 = (long long)mb * BM;
    const int n0 = nb * BN;
    // staging: float4 sq of the stage, rows srow, srow + 32, ... as 32-bit byte offsets from scalar bases that advance
    // with k (vector instructions are what the matrix cores wait for here)
    const int sq = tid & 7, srow = tid >> 3;
    const char* abase = reinterpret_cast<const char*>(p.A + m0 * p.lda);
    const char* wbase = reinterpret_cast<const char*>(static_cast<const float*>(p.W) + (long long)n0 * p.ldw);
    const char* sbase = reinterpret_cast<const char*>(p.scale);
    const int mrows = int(min((long long)BM, p.M - m0)), nrows = min(BN, p.N - n0);
    unsigned ao[APT], wo[WPT], so[APT];
#pragma unroll
    for (int i = 0; i < APT; ++i) {
        const int row = min(srow + 32 * i, mrows - 1);
        ao[i] = unsigned(row * (int)p.lda + 4 * sq) * 4u;
        so[i] = SCALE ? unsigned(int((m0 + row) / p.scale_rows) * p.ld_scale + 4 * sq) * 4u : 0u;
    }
#pragma unroll
    for (int i = 0; i < WPT; ++i) wo[i] = unsigned(min(srow + 32 * i, nrows - 1) * (int)p.ldw + 4 * sq) * 4u;
    f32x4 ra[APT], rw[WPT];
    const auto load = [&](const char* base, unsigned off) { return *reinterpret_cast<const f32x4*>(base + off); };
    const auto fetch_at = [&](int k0, unsigned back) {   // `back`: bytes this lane's float4 is pulled back
#pragma unroll
        for (int i = 0; i < APT; ++i) {
            ra[i] = load(abase + 4ll * k0, ao[i] - back);
            if constexpr (SCALE) ra[i] = load(sbase + 4ll * k0, so[i] - back) * ra[i];
        }
#pragma unroll
        for (int i = 0; i < WPT; ++i) rw[i] = load(wbase + 4ll * k0, wo[i] - back);
        // the loads are issued here, ahead of the stage's matrix work (the scheduler moves them to their first use)
        __builtin_amdgcn_sched_barrier(0);
    };
    const auto fetch = [&](int k0) {   // K % 4 == 0: a float4 is all in or all out; past K: the row's last, not used
        if (k0 >= p.K) return;
        if (k0 + TSTAGE <= p.K) fetch_at(k0, 0u);
        else fetch_at(k0, unsigned(max(k0 + 4 * sq + 4 - p.K, 0)) * 4u);
    };
    // LDS [chunk][row][g][j]: k = 4 j + g of the chunk, so that a fragment read is one float4 of the row
    const int at = (sq >> 2) * ACH + srow * 16 + (sq & 3), wt = (sq >> 2) * WCH + srow * 16 + (sq & 3);
    const auto put = [&](int b) {
#pragma unroll
        for (int i = 0; i < APT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) As[b][at + 512 * i + 4 * e] = ra[i][e];
#pragma unroll
        for (int i = 0; i < WPT; ++i)
            if (BN % 32 == 0 || srow + 32 * i < BN)
#pragma unroll
                for (int e = 0; e < 4; ++e) Ws[b][wt + 512 * i + 4 * e] = rw[i][e];
    };
    // sums of the complete K blocks; -0 + x is x for every x, so the first block's sum is taken as is
    f32x4 tot[WN], blk[WN];
#pragma unroll
    for (int j = 0; j < WN; ++j) tot[j] = f32x4{-0.0f, -0.0f, -0.0f, -0.0f};
    const auto clear = [&] {
#pragma unroll
        for (int j = 0; j < WN; ++j) blk[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    };
    const auto fold = [&] {
#pragma unroll
        for (int j = 0; j < WN; ++j) tot[j] = tot[j] + blk[j];
    };
    const float* afrag = &As[0][(wave * 16 + r) * 16 + 4 * g];
    const float* wfrag = &Ws[0][r * 16 + 4 * g];
    // chunk c of buffer b: NJ k steps
    const auto chunk = [&](int b, int c, auto njc) {
        constexpr int NJ = decltype(njc)::value;
        const f32x4 a = ld4(afrag + b * (2 * ACH) + c * ACH);
        f32x4 w[WN];
#pragma unroll
        for (int j = 0; j < WN; ++j) w[j] = ld4(wfrag + b * (2 * WCH) + c * WCH + j * 256);
#pragma unroll
        for (int q = 0; q < NJ; ++q)
#pragma unroll
            for (int j = 0; j < WN; ++j) blk[j] = mfma4(a[q], w[j][q], blk[j]);
    };
    const std::integral_constant<int, 4> four;
    fetch(0);
    put(0);
    const int nfull = p.K / KBLK;
    for (int b = 0; b < nfull; ++b) {   // whole K blocks: two stages, buffers 0 and 1
        clear();
        __syncthreads();
        fetch(b * KBLK + TSTAGE);
        chunk(0, 0, four);
        chunk(0, 1, four);
        put(1);
        __syncthreads();
        fetch((b + 1) * KBLK);   // past K: clamped, not used
        chunk(1, 0, four);
        chunk(1, 1, four);
        put(0);
        fold();
    }
    int left = p.K - nfull * KBLK;
    if (left) {   // the last, shorter block: exactly K's steps (see steps())
        clear();
        for (int b = 0;; ++b) {
            __syncthreads();
            const bool more = left > TSTAGE;
            if (more) fetch(nfull * KBLK + TSTAGE);
            for (int c = 0; c < 2 && left > 0; ++c, left -= 16) {
                if (left >= 16) chunk(b, c, four);
                else if (left == 12) chunk(b, c, std::integral_constant<int, 3>());
                else if (left == 8) chunk(b, c, std::integral_constant<int, 2>());
                else chunk(b, c, std::integral_constant<int, 1>());
            }
            if (!more) break;
            put(1);
        }
        fold();
    }
    store_strip<WN>(p, swiglu, m0 + wave * 16, n0, g, r, tot);
}

// ------------------------------------------------------------------------------------------------ K blocks over waves
// Small problems (one clip's late layers, 321-row windows, the last rows, SE excitations) do not fill the device
// with whole tiles.  Here the workgroup's W waves share one tile of 16 MT x 16 NT and take its K blocks in turn
// (block b to wave b % W), straight from global memory with a whole block's operands in flight; the block sums meet
// in LDS and are added in order, so the result is bitwise that of the tiled kernel.  Bound by latency: a block is
// one round trip to L2 / HBM and 16 MT NT MFMAs.
template <int MT, int NT, bool SCALE>
__global__ void __launch_bounds__(256) gemm_f32_split_kernel(GemmArgs p, int swiglu, int nkb) {
    constexpr int W = 4;
    extern __shared__ __attribute__((aligned(16))) unsigned char dyn[];
    f32x4* part = reinterpret_cast<f32x4*>(dyn);   // [K block][MT * NT][64]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, r = lane & 15;
    const long long m0 = (long long)blockIdx.x * (16 * MT);
    const int n0 = blockIdx.y * (16 * NT);
    const float *ap[MT], *wp[NT], *sp[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const long long m = min(m0 + 16 * i + r, (long long)p.M - 1);
        ap[i] = p.A + m * p.lda;
        sp[i] = SCALE ? p.scale + (m / p.scale_rows) * p.ld_scale : nullptr;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) wp[j] = static_cast<const float*>(p.W) + (long long)min(n0 + 16 * j + r, p.N - 1) * p.ldw;
    for (int b = wave; b < nkb; b += W) {
        const int k0 = b * KBLK, left = min(KBLK, p.K - k0);
        f32x4 a[4][MT], w[4][NT];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int k = min(k0 + 16 * c + 4 * g, p.K - 4);
#pragma unroll
            for (int i = 0; i < MT; ++i) a[c][i] = ld4(ap[i] + k);
#pragma unroll
            for (int j = 0; j < NT; ++j) w[c][j] = ld4(wp[j] + k);
            if constexpr (SCALE) {
#pragma unroll
                for (int i = 0; i < MT; ++i) a[c][i] = ld4(sp[i] + k) * a[c][i];
            }
        }
        f32x4 acc[MT][NT];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (16 * c >= left) break;
            float at[MT][4], wt[NT][4];
#pragma unroll
            for (int i = 0; i < MT; ++i) transpose4(a[c][i], at[i]);
#pragma unroll
            for (int j = 0; j < NT; ++j) transpose4(w[c][j], wt[j]);
            const auto step = [&](int q) {
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int i = 0; i < MT; ++i) acc[i][j] = mfma4(at[i][q], wt[j][q], acc[i][j]);
            };
            steps(left - 16 * c, step);
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) part[(b * MT * NT + i * NT + j) * 64 + lane] = acc[i][j];
    }
    __syncthreads();
    // tiles (row strip i, U adjacent columns tiles) dealt over the waves; a SwiGLU panel pair stays together
    constexpr int U = NT % 2 == 0 ? 2 : 1;
    for (int t = wave; t < MT * (NT / U); t += W) {
        const int i = t / (NT / U), j0 = (t % (NT / U)) * U;
        f32x4 tot[U];
#pragma unroll
        for (int u = 0; u < U; ++u) tot[u] = part[(i * NT + j0 + u) * 64 + lane];
        for (int b = 1; b < nkb; ++b)
#pragma unroll
            for (int u = 0; u < U; ++u) tot[u] = tot[u] + part[(b * MT * NT + i * NT + j0 + u) * 64 + lane];
        store_strip<U>(p, swiglu, m0 + 16 * i, n0 + 16 * j0, g, r, tot);
    }
}

// ------------------------------------------------------------------------------------------------ launch
template <int WN> void launch_tile(const GemmArgs& p, int swiglu, hipStream_t s) {
    const int mblocks = int(cdiv(p.M, 64)), nblocks = int(cdiv(p.N, 16 * WN));
    const long long blocks = (long long)cdiv(mblocks, XCDS) * XCDS * nblocks;
    if (blocks >= (1ll << 31)) throw std::runtime_error("gemm_f32: grid too large");
    const dim3 grid((unsigned)blocks);
    if (p.scale) hipLaunchKernelGGL((gemm_f32_tile_kernel<WN, true>), grid, dim3(256), 0, s, p, swiglu, mblocks, nblocks);
    else hipLaunchKernelGGL((gemm_f32_tile_kernel<WN, false>), grid, dim3(256), 0, s, p, swiglu, mblocks, nblocks);
}
void launch_tile_wn(int wn, const GemmArgs& p, int swiglu, hipStream_t s) {
    switch (wn) {
    case 1: launch_tile<1>(p, swiglu, s); return;
    case 2: launch_tile<2>(p, swiglu, s); return;
    case 3: launch_tile<3>(p, swiglu, s); return;
    case 4: launch_tile<4>(p, swiglu, s); return;
    case 5: launch_tile<5>(p, swiglu, s); return;
    default: launch_tile<6>(p, swiglu, s); return;
    }
}
template <int MT, int NT> void launch_split(const GemmArgs& p, int swiglu, hipStream_t s) {
    const int nkb = int(cdiv(p.K, KBLK));
    const dim3 grid(cdiv(p.M, 16 * MT), cdiv(p.N, 16 * NT));
    const size_t lds = size_t(nkb) * MT * NT * 1024;
    if (p.scale) hipLaunchKernelGGL((gemm_f32_split_kernel<MT, NT, true>), grid, dim3(256), lds, s, p, swiglu, nkb);
    else hipLaunchKernelGGL((gemm_f32_split_kernel<MT, NT, false>), grid, dim3(256), lds, s, p, swiglu, nkb);
}

struct Plan {
    bool split;
    int mt, nt;   // 16-row and 16-column tiles per workgroup (tiled: 4 x nt)
};
Plan plan(const GemmArgs& p, int swiglu) {
    const int tiles = int(cdiv(p.N, 16)), nkb = int(cdiv(p.K, KBLK));
    // the columns dealt evenly over as few blocks of at most 6 tiles as hold them (SwiGLU panels: pairs of tiles)
    const int nb = int(cdiv(tiles, 6));
    const int wn = swiglu == 2 ? 6 : int(cdiv(tiles, nb));
    // Tiles while they give every CU a workgroup (a short K, whose tiles are quick, from half that), else K blocks over
    // the waves; measured in us, tile / split 2 x 2 / split 1 x 1: 1284 x 2316 x 384 (525 tiles) 41 / 46 / 69, 630 x 2316
    // x 384 (250) 29 / 26 / 37, 1200 x 960 x 160 (190) 10.4 / 13.1 / 16.6, 1200 x 160 x 960 (38) 30 / 12.2 / 14.8,
    // 321 x 384 x 768 (24 tiles, 132 2 x 2s) 29 / 10.8 / 9.7.
    // One block of rows is split however many columns there are, since the split kernel's tiles hold fewer padding rows and
    // have their K blocks in flight at once: tile / split 2 x 2 at 5 x 30000 x 64 31.9 / 5.9, 32 x 30000 x 960 262 / 37, 64 x
    // 100000 x 256 257 / 58.
    const long long wgs = (long long)cdiv(p.M, 64) * nb;
    const bool one = p.M <= 64;
    if (!one && (wgs >= 256 || (nkb <= 3 && wgs >= 128))) return {false, 4, wn};
    // Past 16 K blocks only the smallest tile's block sums fit the LDS.  Its operands are read once per 16 rows and columns,
    // so it is the faster one for few tiles only; tile / split 1 x 1: 5 x 384 x 1100 (24 16 x 16s) 39 / 7.2, 20 x 960 x 2048
    // (120) 68 / 11, 64 x 30000 x 2048 (one block of rows) 549 / 215, 1000 x 384 x 2052 (1512) 70 / 43, 600 x 960 x 2048
    // (2280) 70 / 67, 600 x 960 x 4096 133 / 149, 2000 x 384 x 1100 (3000) 40 / 48.
    if (nkb > 16) {
        const int nt = swiglu == 2 ? 2 : 1;
        if (nkb * nt > 64 || (!one && (long long)cdiv(p.M, 16) * tiles > 1536)) return {false, 4, wn};
        return {true, 1, nt};
    }
    if ((long long)cdiv(p.M, 32) * cdiv(tiles, 2) >= 160) return {true, 2, 2};
    return {true, 1, swiglu == 2 ? 2 : 1};
}

}  // namespace

bool gemm_f32_mc_ok(const GemmArgs& p) {
    const auto al16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    return p.K % 4 == 0 && p.lda % 4 == 0 && p.ldw % 4 == 0 && p.lda >= p.K && p.ldw >= p.K && al16(p.A) && al16(p.W) &&
           (!p.scale || (p.ld_scale % 4 == 0 && al16(p.scale) &&
                         ((long long)p.M / p.scale_rows + 1) * p.ld_scale < (1ll << 30))) &&
           p.lda < (1 << 22) && p.ldw < (1 << 22) &&   // 32-bit offsets inside a tile, a strip and the scale rows
           p.ldc < (1 << 27) && p.ldr < (1 << 27);
}

void gemm_f32_mc(const GemmArgs& p, int swiglu, hipStream_t s) {
    const Plan pl = plan(p, swiglu);
    if (!pl.split) launch_tile_wn(pl.nt, p, swiglu, s);
    else if (pl.mt == 2) launch_split<2, 2>(p, swiglu, s);
    else if (pl.nt == 2) launch_split<1, 2>(p, swiglu, s);
    else launch_split<1, 1>(p, swiglu, s);
}

std::string gemm_f32_mc_kernel(const GemmArgs& p, int swiglu) {
    const Plan pl = plan(p, swiglu);
    return pl.split ? "gemm_f32_split_kernel<" + std::to_string(pl.mt) + "," + std::to_string(pl.nt) + ">"
                    : "gemm_f32_tile_kernel<" + std::to_string(pl.nt) + ">";
}

}  // namespace shv
