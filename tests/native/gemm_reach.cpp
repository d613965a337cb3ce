// The weights that the wide pointwise GEMM's lanes read (shield-sisa_amd/csrc/gemm_reach.hpp) lie in their row, whole and in
// place, for every K that the kernel takes.
#include <cstdio>

#include "../../shield-sisa_amd/csrc/gemm_reach.hpp"

int main() {
    int bad = 0;
    for (int K = 8; K <= 256; K += 8)
        for (int ks = 0; ks < (K + 31) / 32; ++ks)
            for (int g = 0; g < 4; ++g) {
                const bool in = 32 * ks + 8 * g < K;
                const int k = 8 * g + shv::wide_step((K + 31) / 32, ks, g, in);
                if (k < 0 || k + 8 > K || (in && k != 32 * ks + 8 * g)) {
                    std::printf("K %d step %d group %d reads from %d\n", K, ks, g, k);
                    ++bad;
                }
            }
    return bad ? 1 : 0;
}
