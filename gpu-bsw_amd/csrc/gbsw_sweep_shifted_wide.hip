// gbsw_sweep_shifted_wide.hip -- sweep kernels with one pair per wave: byte tables that
// hold the scores from the smallest one up (KernelArgs::shift).
#include "gbsw_sweep.hpp"

namespace gbsw {

template <int PF>
static const void* shifted_wide(int kind, int K)
{
    if ((kind & 0xFF) != kSplitF16) return (const void*)&k_sweep<Sweep16Shifted, 64, PF, false>;
    switch (K) {
#define GBSW_CASE(k) case k: return (const void*)&k_sweep_split<Sweep16Shifted, 64, k, PF>;
        GBSW_SWEEP_K64_SPLIT(GBSW_CASE)
#undef GBSW_CASE
    default: return nullptr;
    }
}

const void* sweep_kernel_shifted_wide(int kind, int K)
{
    return (kind & kRegTables) ? shifted_wide<kProfRegs>(kind, K) : shifted_wide<kProfBytes>(kind, K);
}

} // namespace gbsw
