// The bytes that the crop kernel's word loads touch, worked out from its own plans, choice of kernel and word counts
// (shield-sisa_amd/csrc/crop_plan.hpp): over frames of any size, stored with the tightest strides and nothing after the last
// pixel, no load may end past its plane.  A row of the plane's last pixel row (I420: last chroma row) is read byte by byte,
// and so is everything in variant 0.  Beside it: the LDS ring holds a chunk's patch columns, and the I420 conversion equals
// its 16-bit form.
#include <cstdio>

#include "../../shield-sisa_amd/csrc/crop_plan.hpp"

using namespace shv;

// bytes past the end of the worst plane (<= 0: none) of a w x h frame
static long long reach(int w, int h, bool i420) {
    CanvasGeo g;
    PlanHost p;
    if (!canvas_geo(w, h, g) || !make_plan(w, h, g.new_w, g.new_h, g.mode == 2 ? 1 : 3, p)) return -1;   // refused
    if (crop_variant(p.K, p.fin, p.sw, i420) == 0) return -1;
    const int K = p.K, cw = (w + 1) / 2, ch = (h + 1) / 2;
    int x = 0;
    for (int o : p.xoff) x = o > x ? o : x;
    long long worst = -1;
    for (int y = 0; y < g.new_h; ++y) {
        const int* rows = p.ysi.data() + size_t(y) * K;
        if (i420 ? rows[K - 1] / 2 == ch - 1 : rows[K - 1] == h - 1) continue;
        for (int j = 0; j < K; ++j) {
            const long long r = rows[j];
            if (i420) {
                worst = std::max(worst, r * w + x + 4 * load_words(K) - (long long)w * h);
                worst = std::max(worst, r / 2 * cw + x / 2 + 4 * load_words(chroma_samples(K)) - (long long)cw * ch);
            } else {
                worst = std::max(worst, r * 3 * w + 3 * x + 4 * load_words(3 * K) - 3ll * w * h);
            }
        }
    }
    return worst;
}

static int sat16(int v) { return v < -32768 ? -32768 : (v > 32767 ? 32767 : v); }

int main() {
    int frames = 0, bad = 0;
    // every I420 pixel against the 16-bit arithmetic with its saturations
    const int yc = 9539, vr = 13075, ub = 16525, ug = -3209, vg = -6660;
    for (int y = 0; y < 256; ++y)
        for (int u = 0; u < 256; ++u)
            for (int v = 0; v < 256; ++v) {
                const int yy = (int(short((y << 3) - 128)) * yc) >> 16, up = sat16((u << 3) - 1024), vp = sat16((v << 3) - 1024);
                const int r = yuv_sat8(sat16(yy + ((vp * vr) >> 16))), b = yuv_sat8(sat16(yy + ((up * ub) >> 16)));
                const int g = yuv_sat8(sat16(yy + sat16(((up * ug) >> 16) + ((vp * vg) >> 16))));
                const int l = yuv_luma(y);
                if (yuv_sat8(l + yuv_red(v)) != r || yuv_sat8(l + yuv_green(u, v)) != g || yuv_sat8(l + yuv_blue(u)) != b) ++bad;
            }
    if (bad) std::printf("%d I420 pixels differ\n", bad);
    const auto check = [&](int w, int h) {
        for (int i420 = 0; i420 < 2; ++i420, ++frames) {
            const long long r = reach(w, h, i420);
            if (r > 0 && ++bad <= 20) std::printf("%s %dx%d: %lld bytes past a plane\n", i420 ? "I420" : "RGB", w, h, r);
        }
    };
    for (int w = 1; w <= 24; ++w)
        for (int h = 1; h <= 2900; h = h < 64 || (h > 700 && h < 740) ? h + 1 : h + 37) check(w, h);
    for (int h = 1; h <= 12; ++h)
        for (int w = 25; w <= 6000; w += 131) check(w, h);
    for (int s = 1; s <= 40; ++s) check(160 * s, 90 * s), check(90 * s, 160 * s), check(160 * s + 1, 90 * s + 1);
    // the LDS ring holds the patch columns of every chunk of output columns
    for (int w4 = 80; w4 <= 320; ++w4)
        for (int chunks = 1; chunks <= 4; chunks *= 2) {
            const int pw = 4 * w4, cols = CROP_W / chunks;
            PlanHost p;
            if (!make_plan(pw, 4 * 45, CROP_W, CROP_H, 3, p) || p.K > CROP_KMAX) {
                ++bad;
                continue;
            }
            for (int c = 0; c < CROP_W; c += cols) {
                const int need = p.xoff[size_t(c + cols - 1)] + p.K - p.xoff[size_t(c)];
                if (need > ring_width(pw, cols) && ++bad <= 20)
                    std::printf("patch %d: %d columns, room for %d\n", pw, need, ring_width(pw, cols));
            }
        }
    std::printf("%d frames, %d out of range\n", frames, bad);
    return bad ? 1 : 0;
}
