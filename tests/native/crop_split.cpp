// Workgroups of a call's crops (shield-sisa_amd/csrc/crop_plan.hpp): whatever the kernel and however few the crops, about one
// for each of the device's 256 CUs; every split covers the 180 x 320 outputs in whole quads of columns.
#include <cstdio>

#include "../../shield-sisa_amd/csrc/crop_plan.hpp"

int main() {
    int bad = 0;
    for (int v = 0; v < shv::CROP_VARIANTS; ++v)
        for (int new_w = 1; new_w <= 1280; new_w = new_w < 4 ? new_w + 1 : 2 * new_w)
            for (int n = 1; n <= 3000; ++n) {
                const shv::CropSplit s = shv::crop_split(n, v, new_w);
                const int bands = s.band > 0 ? (shv::CROP_H + s.band - 1) / s.band : 0;
                if (bands < 1 || s.chunks < 1 || shv::CROP_W % (4 * s.chunks) || (long long)n * bands * s.chunks < 240) {
                    if (++bad <= 20) std::printf("variant %d, %d crops: bands of %d rows, %d chunks\n", v, n, s.band, s.chunks);
                }
            }
    return bad ? 1 : 0;
}
