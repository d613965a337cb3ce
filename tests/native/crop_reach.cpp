// The bytes that the crop kernel's word loads touch, worked out from its own plans, choice of kernel and word counts
// (shield-sisa_amd/csrc/crop_plan.hpp): over frames of any size, stored with the tightest strides and nothing after the last
// pixel, no load may end past its plane.  A row of the plane's last pixel row (I420: last chroma row) is read byte by byte,
// and so is everything in variant 0.
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

int main() {
    int frames = 0, bad = 0;
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
    std::printf("%d frames, %d out of range\n", frames, bad);
    return bad ? 1 : 0;
}
