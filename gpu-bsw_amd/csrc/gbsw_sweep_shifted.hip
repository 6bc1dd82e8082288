// gbsw_sweep_shifted.hip -- sweep kernels with four and eight pairs per wave: byte tables
// that hold the scores from the smallest one up (KernelArgs::shift).
#include "gbsw_sweep_pairs.hpp"

namespace gbsw {

const void* sweep_kernel_shifted(int kind)
{
    const bool wide = (kind & kWideLanes) != 0;
    if (kind & kHalfPairs)
        return wide ? (const void*)&k_sweep_pairs<Sweep16Shifted, true> : (const void*)&k_sweep_pairs<Sweep16Shifted, false>;
    if (kind & kRegTables)
        return wide ? (const void*)&k_sweep<Sweep16Shifted, 16, kProfRegs, true>
                    : (const void*)&k_sweep<Sweep16Shifted, 16, kProfRegs, false>;
    return wide ? (const void*)&k_sweep<Sweep16Shifted, 16, kProfBytes, true>
                : (const void*)&k_sweep<Sweep16Shifted, 16, kProfBytes, false>;
}

} // namespace gbsw
