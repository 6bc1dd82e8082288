// gbsw_sweep_regs.hip -- sweep kernels: register tables (at most four residue codes).
#include "gbsw_sweep.hpp"

namespace gbsw {

#define GBSW_SWEEP_PF kProfRegs
#ifndef GBSW_SWEEP_K16
#define GBSW_SWEEP_K16(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(10) X(12) X(14) X(16)
#endif
#ifndef GBSW_SWEEP_SPLIT_K16
#define GBSW_SWEEP_SPLIT_K16(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(10) X(12) X(14) X(16)
#endif

const void* sweep_kernel_regs(bool split, bool wide, int K)
{
    if (wide) return nullptr;
#define GBSW_SWEEP_G 16
    if (split) {
        switch (K) {
            GBSW_SWEEP_SPLIT_K16(GBSW_SWEEP_SPLIT_CASE)
        default: return nullptr;
        }
    }
    switch (K) {
        GBSW_SWEEP_K16(GBSW_SWEEP_CASE)
    default: return nullptr;
    }
#undef GBSW_SWEEP_G
}

} // namespace gbsw
