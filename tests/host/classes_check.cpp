// CPU check of the length classes, sort keys and LDS sizes of the sweep kernels
// (gbsw_kernel_args.hpp) over every accepted length.  Prints the first failure, or "ok".
#include <cstdio>

#include "../../gpu-bsw_amd/csrc/gbsw_kernel_args.hpp"

using namespace gbsw;

#define CHECK(x)                                          \
    do {                                                  \
        if (!(x)) {                                       \
            std::printf("m %d: %s\n", m, #x);             \
            return 1;                                     \
        }                                                 \
    } while (0)

int main()
{
    for (int m = 0; m <= 65000; ++m) {
        const int c = length_class(m), f = fine_class(m);
        CHECK(c >= 0 && c < kClasses && f >= 0 && f < kFineClasses);
        if (m) {
            // no gaps and in order, and a fine class never spans two classes
            const int pc = length_class(m - 1), pf = fine_class(m - 1);
            CHECK(c == pc || c == pc + 1);
            CHECK(f == pf || f == pf + 1);
            CHECK(c == pc || f == pf + 1);
        }
        if (m >= 1 && m <= kPairsCols) {
            // one geometry per class: columns per lane with eight and with four pairs per wave
            const int k16 = (m + 15) / 16, k32 = (m + 31) / 32;
            CHECK((k16 < 2 ? 2 : k16) == f + 2);
            CHECK((k32 < 2 ? 2 : k32) == c + 2);
        }
        // the key: class and rows, the class in the upper bits
        CHECK((((unsigned)(kFineClasses - 1 - f) << kRowBits) | ((1u << kRowBits) - 1u)) < (1u << kSortBits));
    }
    for (int alpha = 1; alpha <= kRegAlpha; ++alpha) { // 16 waves of eight pairs fit a CU's 160 KiB
        const int m = alpha;
        CHECK(pairs_lds(16, alpha).total <= 160 * 1024 / 16);
    }
    for (int alpha = 1; alpha <= kMaxAlpha; ++alpha)
        for (int K = 1; K <= 16; ++K) {
            const int m = alpha;
            for (int form = kProfRegs; form <= kProfWords; ++form) {
                const SweepLds L = sweep_lds(16, K, form, alpha, 4);
                CHECK(L.ring_bnd_off <= L.group_bytes && L.group_off % 128 == 0 && L.group_bytes % 128 == 0);
                const SweepLds W = sweep_lds(64, K, form, alpha, 8);
                CHECK(W.ring_bnd_off + (sweep_ring(64) + kSweepUnroll) * 8 <= W.group_bytes && W.ring_bnd_off % 8 == 0);
            }
        }
    std::printf("ok\n");
    return 0;
}
