// SHIELD-A frontend kernels for gfx950 (the reference: engine/audio/frontend.cpp): the log-mel frames of a 10 s
// window and the frequency-attention pooling.  The CNN's stem and its blocks' expand and depthwise layers are expdw.hip's,
// the 1x1 projections and the token projection GEMMs of the engine's tiers.  Activations are fp32 in HBM, image layout [time][freq][channel].
//
// Per element these kernels perform the reference's IEEE operations in its order (the reference is compiled with
// -ffp-contract=off, and so is this file): the radix-2 FFT's butterflies, the power spectrum, the filterbank fma
// chain, the softmax's running sum.  The device's exp and log (softmax, mel energies) are within an ulp or two of glibc's.
#include "dev_common.hpp"
#include "kernels.hpp"

#include <stdexcept>

namespace shv {
namespace {

inline unsigned int cdiv(long long a, long long b) { return (unsigned int)((a + b - 1) / b); }

// waits for the wave's own LDS accesses: LDS executes one wave's instructions in order, so after this every lane
// sees what every lane of the wave wrote before
__device__ __forceinline__ void wave_lds_sync() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// ---------------------------------------------------------------------------------------------------- log-mel
// One wave per frame, four frames per workgroup.  Frame t's 400 windowed samples pcm[t * 160 + 56 + j] * window[j]
// go to the bit-reversed slots of a 512-point buffer (the rest zero), nine radix-2 stages run in place with the
// twiddles e^{-2 pi i k / 512} (host-computed in double, rounded to float), then |X_k|^2 for k <= 256, each mel bin's
// fma chain over its filter's nonzero taps in increasing k, and (log(e + 1e-6) - mean) / std
// (frontend.cpp:245-256).
constexpr int MEL_WAVES = 4;

__global__ void __launch_bounds__(64 * MEL_WAVES) audio_mel_kernel(const float* __restrict__ pcm, long long stride,
                                                                   AudioMelTables tb, float* __restrict__ mel) {
    __shared__ float re[MEL_WAVES][512], im[MEL_WAVES][512];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t = blockIdx.x * MEL_WAVES + wave;
    if (t >= kAudioMelFrames) return;   // wave-uniform; no workgroup barrier follows
    const long long win = blockIdx.y;
    float* R = re[wave];
    float* I = im[wave];
    for (int i = lane; i < 512; i += 64) {
        R[i] = 0.0f;
        I[i] = 0.0f;
    }
    wave_lds_sync();
    const float* x = pcm + win * stride + (long long)t * 160;
    for (int n = 56 + lane; n < 456; n += 64) R[__builtin_bitreverse32(unsigned(n)) >> 23] = x[n] * tb.window[n - 56];
    wave_lds_sync();
#pragma unroll 1
    for (int lh = 0; lh < 9; ++lh) {   // half = 2^lh, size = 2 half, twiddle step 256 / half
        const int half = 1 << lh;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int b = lane + 64 * q;                  // butterfly 0..255
            const int j = b & (half - 1), a = ((b >> lh) << (lh + 1)) + j, c = a + half;
            const int k = j << (8 - lh);
            const float wr = tb.wr[k], wi = tb.wi[k];
            const float rb = R[c], ib = I[c], ra = R[a], ia = I[a];
            const float r = wr * rb - wi * ib, ii = wr * ib + wi * rb;
            R[a] = ra + r;
            I[a] = ia + ii;
            R[c] = ra - r;
            I[c] = ia - ii;
        }
        wave_lds_sync();
    }
    for (int k = lane; k <= 256; k += 64) R[k] = R[k] * R[k] + I[k] * I[k];
    wave_lds_sync();
    float* out = mel + (win * kAudioMelFrames + t) * kAudioMelBins;
    for (int m = lane; m < kAudioMelBins; m += 64) {
        float v = 0.0f;
        for (int e = tb.fb_off[m]; e < tb.fb_off[m + 1]; ++e) v = __builtin_fmaf(tb.fb_w[e], R[tb.fb_k[e]], v);
        out[m] = (logf(v + 1e-6f) - tb.mean[m]) / tb.stdv[m];
    }
}

// ---------------------------------------------------------------------------------------------------- attention
// Frequency attention over the [125][20][192] image (frontend.cpp:222-231), one wave per time step: the 20 logits
// (an fma chain from +0 over the 192 channels, then + bias), their softmax (running max, exp(l - max), the sum in
// frequency order, division), and pooled[c] = sum over f of v * a_f from +0 in frequency order.
__global__ void __launch_bounds__(256) audio_freq_pool_kernel(const float* __restrict__ h, const float* __restrict__ w,
                                                              float bias, float* __restrict__ pooled, long long steps) {
    __shared__ float a[4][kAudioCnnFreq];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long step = (long long)blockIdx.x * 4 + wave;
    if (step >= steps) return;   // wave-uniform
    const float* v = h + step * (kAudioCnnFreq * kAudioCnnCh);
    float l = 0.0f;
    if (lane < kAudioCnnFreq) {
        const float* row = v + lane * kAudioCnnCh;
        for (int c = 0; c < kAudioCnnCh; ++c) l = __builtin_fmaf(row[c], w[c], l);
        l = l + bias;
        a[wave][lane] = l;
    }
    wave_lds_sync();
    float mx = -__builtin_inff();
    for (int f = 0; f < kAudioCnnFreq; ++f) mx = fmaxf(mx, a[wave][f]);
    wave_lds_sync();
    const float e = expf(l - mx);
    if (lane < kAudioCnnFreq) a[wave][lane] = e;
    wave_lds_sync();
    float sum = 0.0f;
    for (int f = 0; f < kAudioCnnFreq; ++f) sum = sum + a[wave][f];
    wave_lds_sync();
    if (lane < kAudioCnnFreq) a[wave][lane] = e / sum;
    wave_lds_sync();
    for (int c = lane; c < kAudioCnnCh; c += 64) {
        float p = 0.0f;
        for (int f = 0; f < kAudioCnnFreq; ++f) p = p + v[f * kAudioCnnCh + c] * a[wave][f];
        pooled[step * kAudioCnnCh + c] = p;
    }
}

}  // namespace

void launch_audio_mel(const float* pcm, long long stride, int n, const AudioMelTables& tb, float* mel, hipStream_t s) {
    if (n <= 0) return;
    if (!pcm || !mel || stride < kAudioWindowSamples) throw std::runtime_error("audio mel: bad PCM or window stride");
    hipLaunchKernelGGL(audio_mel_kernel, dim3(cdiv(kAudioMelFrames, MEL_WAVES), (unsigned)n), dim3(64 * MEL_WAVES), 0,
                       s, pcm, stride, tb, mel);
}

void launch_audio_freq_pool(const float* h, const float* w, float bias, float* pooled, int n, hipStream_t s) {
    if (n <= 0) return;
    const long long steps = (long long)n * kAudioTokensPerWindow;
    hipLaunchKernelGGL(audio_freq_pool_kernel, dim3(cdiv(steps, 4)), dim3(256), 0, s, h, w, bias, pooled, steps);
}

}  // namespace shv
