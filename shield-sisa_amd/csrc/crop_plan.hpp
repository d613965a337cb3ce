// Host side of the face crops (crop.hip), free of the HIP runtime: the resize plans (taps, weights, coefficients, in the
// reference's double / float arithmetic), the canvas geometry, and the choice of kernel.
#pragma once
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <vector>

namespace shv {

constexpr int CROP_W = 320, CROP_H = 180, COEF_BITS = 11, COEF_SCALE = 1 << COEF_BITS;
constexpr int CROP_KMAX = 5;    // canvas rows and columns per output pixel (scales up to 4)

// how a column pass ends (rounding after a scale, 1 where there is none; the 2 x 2 blocks' and the linear resize's integer
// forms have K = 2)
enum Finish { FIN_SCALE = 0, FIN_QUARTER = 1, FIN_LINEAR = 2 };

inline long py_round(double v) { return long(std::nearbyint(v)); }   // Python round(): half to even
inline int rint_f(float v) { return int(std::nearbyintf(v)); }

struct Tap {
    int d, s;
    float w;
};
// OpenCV's area taps for one axis (computeResizeAreaTab): output cell [d scale, (d + 1) scale) of the source,
// partial source pixels weighted by their covered fraction of the cell
inline std::vector<Tap> area_taps(int ssize, int dsize, double scale) {
    std::vector<Tap> t;
    for (int d = 0; d < dsize; ++d) {
        const double f1 = d * scale, f2 = f1 + scale;
        const double cell = std::min(scale, ssize - f1);
        int s1 = int(std::ceil(f1)), s2 = int(std::floor(f2));
        s2 = std::min(s2, ssize - 1);
        s1 = std::min(s1, s2);
        if (s1 - f1 > 1e-3) t.push_back({d, s1 - 1, float((s1 - f1) / cell)});
        for (int s = s1; s < s2; ++s) t.push_back({d, s, float(1.0 / cell)});
        if (f2 - s2 > 1e-3) t.push_back({d, s2, float(std::min(std::min(f2 - s2, 1.0), cell) / cell)});
    }
    return t;
}

struct PlanHost {
    int fin = FIN_SCALE, K = 1, sw = 0, sh = 0;
    float fscale = 1.0f;
    std::vector<int> xoff, ysi;
    std::vector<float> xw, yw;
};

// Taps per output (consecutive source pixels in order) as K-wide tables.  Zero weights fill the places an output has no
// tap: columns are K neighbouring pixels, pulled back where they would pass the source's end (a source narrower than K
// takes the pixel-by-pixel path); rows repeat the last.
inline void set_taps(PlanHost& p, const std::vector<std::vector<Tap>>& cols, const std::vector<std::vector<Tap>>& rows) {
    p.K = 1;
    for (const auto& c : cols) p.K = std::max(p.K, int(c.size()));
    for (const auto& r : rows) p.K = std::max(p.K, int(r.size()));
    for (const auto& c : cols) {
        const int off = std::max(0, std::min(c.front().s, p.sw - p.K));
        p.xoff.push_back(off);
        std::vector<float> w(size_t(p.K), 0.0f);
        for (const Tap& t : c) w[size_t(t.s - off)] = t.w;
        p.xw.insert(p.xw.end(), w.begin(), w.end());
    }
    for (const auto& r : rows)
        for (int k = 0; k < p.K; ++k) {
            const Tap& t = r[size_t(std::min(k, int(r.size()) - 1))];
            p.ysi.push_back(t.s);
            p.yw.push_back(k < int(r.size()) ? t.w : 0.0f);
        }
}
inline std::vector<std::vector<Tap>> by_output(const std::vector<Tap>& taps, int n) {
    std::vector<std::vector<Tap>> o(static_cast<size_t>(n));
    for (const Tap& t : taps) o[size_t(t.d)].push_back(t);
    return o;
}
inline std::vector<std::vector<Tap>> blocks(int n, int size) {   // `size` source pixels of weight 1 each
    std::vector<std::vector<Tap>> o(static_cast<size_t>(n));
    for (int d = 0; d < n; ++d)
        for (int k = 0; k < size; ++k) o[size_t(d)].push_back({d, d * size + k, 1.0f});
    return o;
}

// interpolation: 1 INTER_LINEAR, 3 INTER_AREA (OpenCV codes); false where the reference has no plan either
inline bool make_plan(int sw, int sh, int dw, int dh, int interpolation, PlanHost& p) {
    p = PlanHost();
    p.sw = sw; p.sh = sh;
    if (sw <= 0 || sh <= 0 || dw <= 0 || dh <= 0) return false;
    if (sw == dw && sh == dh) {   // copy
        set_taps(p, blocks(dw, 1), blocks(dh, 1));
        return true;
    }
    const double inv_x = double(dw) / sw, inv_y = double(dh) / sh;
    const double scale_x = 1.0 / inv_x, scale_y = 1.0 / inv_y;
    const int isx = int(std::nearbyint(scale_x)), isy = int(std::nearbyint(scale_y));
    const bool fast = std::abs(scale_x - isx) < DBL_EPSILON && std::abs(scale_y - isy) < DBL_EPSILON;
    if (interpolation == 1 && fast && isx == 2 && isy == 2) interpolation = 3;
    if (interpolation == 3) {
        if (!(scale_x >= 1 && scale_y >= 1)) return false;
        if (fast && sw == isx * dw && sh == isy * dh) {
            if (isx == 2 && isy == 2) p.fin = FIN_QUARTER;
            else p.fscale = 1.f / float(isx * isy);
            set_taps(p, blocks(dw, isx), blocks(dh, isy));
            return true;
        }
        set_taps(p, by_output(area_taps(sw, dw, scale_x), dw), by_output(area_taps(sh, dh, scale_y), dh));
        return true;
    }
    if (interpolation != 1) return false;
    p.fin = FIN_LINEAR;
    std::vector<std::vector<Tap>> cols(static_cast<size_t>(dw)), rows(static_cast<size_t>(dh));
    int lxmax = dw;
    for (int dx = 0; dx < dw; ++dx) {
        float fx = float((dx + 0.5) * scale_x - 0.5);
        int sx = int(std::floor(fx));
        fx -= float(sx);
        if (sx < 0) { fx = 0.f; sx = 0; }
        if (sx + 1 >= sw) {
            lxmax = std::min(lxmax, dx);
            if (sx >= sw - 1) { fx = 0.f; sx = sw - 1; }
        }
        if (dx < lxmax) {
            const int a0 = std::max(-32768, std::min(32767, rint_f((1.f - fx) * COEF_SCALE)));
            const int a1 = std::max(-32768, std::min(32767, rint_f(fx * COEF_SCALE)));
            cols[size_t(dx)] = {{dx, sx, float(a0)}, {dx, sx + 1, float(a1)}};
        } else {
            cols[size_t(dx)] = {{dx, sx, float(COEF_SCALE)}};
        }
    }
    for (int dy = 0; dy < dh; ++dy) {
        float fy = float((dy + 0.5) * scale_y - 0.5);
        const int sy = int(std::floor(fy));
        fy -= float(sy);
        const int b0 = std::max(-32768, std::min(32767, rint_f((1.f - fy) * COEF_SCALE)));
        const int b1 = std::max(-32768, std::min(32767, rint_f(fy * COEF_SCALE)));
        const auto clip = [&](int y) { return y >= 0 ? (y < sh ? y : sh - 1) : 0; };
        rows[size_t(dy)] = {{dy, clip(sy), float(b0)}, {dy, clip(sy + 1), float(b1)}};
    }
    set_taps(p, cols, rows);
    return true;
}

// ffmpeg's yuv2rgb coefficients for BT.601 limited range (contrast = saturation = 1 << 16, brightness 0), rounded to 16 bits
// as av_clip_int16((x + 2^15) >> 16): Y 76309 (= 65536 * 255 / 219) and the inverse-table entries 104597 (V->R), 132201
// (U->B), -25675 (U->G), -53279 (V->G), each times 2^13.  The reference works in 16 bits with saturation: (8 y - 128) Y >> 16,
// (8 c - 1024) C >> 16 per chroma table, sums saturated.  No sum of these reaches 16 bits (8-bit operands), so only the last
// one, to 8 bits, is left; as compile-time constants a term is one multiply-add and one shift.
constexpr int yuv_round16(long long f) { return int((f + (1 << 15)) >> 16); }
constexpr int YUV_Y = yuv_round16((65536LL * 255 / 219) * (1 << 13)), YUV_VR = yuv_round16(104597LL * (1 << 13)),
              YUV_UB = yuv_round16(132201LL * (1 << 13)), YUV_UG = yuv_round16(-25675LL * (1 << 13)),
              YUV_VG = yuv_round16(-53279LL * (1 << 13));
constexpr int yuv_luma(int y) { return (y * (8 * YUV_Y) - 128 * YUV_Y) >> 16; }
constexpr int yuv_term(int c, int coeff) { return (c * (8 * coeff) - 1024 * coeff) >> 16; }
constexpr int yuv_red(int v) { return yuv_term(v, YUV_VR); }
constexpr int yuv_green(int u, int v) { return yuv_term(u, YUV_UG) + yuv_term(v, YUV_VG); }
constexpr int yuv_blue(int u) { return yuv_term(u, YUV_UB); }
constexpr int yuv_sat8(int v) { return v < 0 ? 0 : (v > 255 ? 255 : v); }

// canvas geometry of a w x h frame (geometry.cpp:77-88): scale min(720/h, 1280/w), centred, mode 0 copy /
// 1 shrink (area) / 2 enlarge (linear)
struct CanvasGeo {
    int new_w, new_h, left, top, mode;
};
inline bool canvas_geo(int w, int h, CanvasGeo& g) {
    if (w <= 0 || h <= 0) return false;
    const double scale = std::min(720.0 / h, 1280.0 / w);
    g.new_h = int(std::max(1L, py_round(h * scale)));
    g.new_w = int(std::max(1L, py_round(w * scale)));
    if (g.new_w > 1280 || g.new_h > 720) return false;
    g.left = (1280 - g.new_w) / 2;
    g.top = (720 - g.new_h) / 2;
    g.mode = (g.new_h == h && g.new_w == w) ? 0 : (scale < 1 ? 1 : 2);
    return true;
}

// The launches take the crops of one canvas resize each: K taps and finish, or (0) whatever else.
struct Variant { int K, fin; };
constexpr Variant kVariants[] = {{0, FIN_SCALE}, {1, FIN_SCALE}, {2, FIN_SCALE}, {2, FIN_QUARTER}, {2, FIN_LINEAR},
                                 {3, FIN_SCALE}, {4, FIN_SCALE}, {5, FIN_SCALE}, {6, FIN_SCALE}, {7, FIN_SCALE},
                                 {8, FIN_SCALE}};
constexpr int CROP_VARIANTS = 11;

// What an unrolled kernel reads of a source row for the K pixels from a column on: whole words, so up to three bytes past
// them.  Those lie in the next row, which is there: rows of the plane's last pixel row (I420: last chroma row) are read byte
// by byte.  That takes a next row of three bytes at least: any RGB row, and an I420 row of three chroma samples (the
// chroma words start at the sample of an odd column too).
constexpr int load_words(int bytes) { return (bytes + 3) / 4; }
constexpr int chroma_samples(int K) { return K / 2 + 1; }   // under K pixels from any column
inline int crop_variant(int K, int fin, int sw, bool i420) {   // of a plan over frames sw wide
    if (sw < K || (i420 && (sw + 1) / 2 < 3)) return 0;
    int k = CROP_VARIANTS - 1;
    while (k > 0 && !(K == kVariants[k].K && fin == kVariants[k].fin)) --k;
    return k;
}

// How the crops of one kernel (variant) are split in a call of n, frames resized to new_w columns: bands of `band` output
// rows, and 1, 2 or 4 chunks of their columns.  A band or chunk computes a canvas row or a few columns again, but a workgroup
// walks its rows one after another: few crops want many short ones.  Calls in us: one crop of a 1920 x 1080 frame RGB 36 in
// bands of 3 rows, 25 in 1 row x 2 chunks (I420 56, 27), 4 RGB 40 in 3 rows, 34 in 1, 8 RGB 51 in 3, 46 in 2, 50 in 1, 40 RGB
// 116 in 3, 136 in 1.  7680 x 4320 I420 (6 taps): 4 crops 217 in 1 row, 185 in 3 x 2 chunks, 10 crops 524 in 3, 449 in 3 x 2.
// More than 8 taps: one crop of 9000 x 5000 RGB 293 in 1 x 2, 225 in 1 x 4, 20 of 20000 x 100 1,606 in 3, 709 in 1 x 4, but 20
// of 100 x 20000 (4 live columns) 386 in 3, 1,638 in 1 x 4.
struct CropSplit { int band, chunks; };
inline CropSplit crop_split(int n, int variant, int new_w) {
    if (variant == 0 && new_w >= CROP_W) return {1, 4};   // 81 taps a pixel and more: as many threads as there are pixels
    if (kVariants[variant].K > CROP_KMAX && n > 1 && n <= 16) return {3, 2};
    const int bands = n <= 4 ? 180 : n <= 8 ? 90 : std::max(12, std::min(60, (6144 + n - 1) / n));
    return {(CROP_H + bands - 1) / bands, n <= 2 ? 2 : 1};
}
// Most patch columns under `cols` output columns of a patch pw wide: their cells and a pixel on either side, or the K
// pixels to which the last columns' taps are pulled back.
inline int ring_width(int pw, int cols) { return std::min(pw, (cols * pw + CROP_W - 1) / CROP_W + CROP_KMAX + 1); }

}  // namespace shv
