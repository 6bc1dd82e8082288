// gbsw_sweep_bytes.hip -- sweep kernels with four pairs per wave: byte profile.
#include "gbsw_sweep.hpp"

namespace gbsw {

const void* sweep_kernel_bytes(int kind, int)
{
    return (kind & kWideLanes) ? (const void*)&k_sweep<Sweep16, 16, kProfBytes, true> : (const void*)&k_sweep<Sweep16, 16, kProfBytes, false>;
}

} // namespace gbsw
