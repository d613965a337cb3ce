// Host side of the face crops (crop.hip), free of the HIP runtime: the resize plans (taps, weights, coefficients, in the
// reference's double / float arithmetic), the canvas geometry, and the choice of kernel.
#pragma once
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <vector>

namespace shv {

constexpr int CROP_W = 320, CROP_H = 180, COEF_BITS = 11, COEF_SCALE = 1 << COEF_BITS;
constexpr int CROP_KMAX = 5;    // source pixels per axis of the unrolled kernels (scales up to 4)

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
                                 {3, FIN_SCALE}, {4, FIN_SCALE}, {5, FIN_SCALE}};
constexpr int CROP_VARIANTS = 8;

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

}  // namespace shv
