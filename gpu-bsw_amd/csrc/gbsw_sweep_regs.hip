// gbsw_sweep_regs.hip -- sweep kernels with four pairs per wave: register tables (at most four residue codes).
#include "gbsw_sweep.hpp"

namespace gbsw {

const void* sweep_kernel_regs(int kind, int)
{
    return (kind & kWideLanes) ? (const void*)&k_sweep<Sweep16, 16, kProfRegs, true> : (const void*)&k_sweep<Sweep16, 16, kProfRegs, false>;
}

} // namespace gbsw
