// gbsw_sweep_int32.hip -- sweep kernels with int32 cells (16-bit profile): pairs whose
// score left the 16-bit range, one pair per wave or split over several.
#include "gbsw_sweep.hpp"

namespace gbsw {

const void* sweep_kernel_int32(int kind, int K)
{
    if (!(kind & kSplitStrips)) return (const void*)&k_sweep<Sweep32, 64, kProfWords, false>;
    switch (K) {
#define GBSW_CASE(k) case k: return (const void*)&k_sweep_split<Sweep32, 64, k, kProfWords>;
        GBSW_SWEEP_K32(GBSW_CASE)
#undef GBSW_CASE
    default: return nullptr;
    }
}

} // namespace gbsw
