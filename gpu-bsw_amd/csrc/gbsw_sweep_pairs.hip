// gbsw_sweep_pairs.hip -- the sweep kernel with eight pairs per wave (register tables).
#include "gbsw_sweep_pairs.hpp"

namespace gbsw {

const void* sweep_kernel_pairs(int kind)
{
    return (kind & kWideLanes) ? (const void*)&k_sweep_pairs<Sweep16, true> : (const void*)&k_sweep_pairs<Sweep16, false>;
}

} // namespace gbsw
