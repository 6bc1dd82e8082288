// gbsw_sweep_bytes_wide.hip -- sweep kernels with one pair per wave: byte profile.
#include "gbsw_sweep.hpp"

namespace gbsw {

const void* sweep_kernel_bytes_wide(int kind, int K)
{
    if ((kind & 0xFF) != kSplitF16) return (const void*)&k_sweep<Sweep16, 64, kProfBytes, false>;
    switch (K) {
#define GBSW_CASE(k) case k: return (const void*)&k_sweep_split<Sweep16, 64, k, kProfBytes>;
        GBSW_SWEEP_K64_SPLIT(GBSW_CASE)
#undef GBSW_CASE
    default: return nullptr;
    }
}

} // namespace gbsw
