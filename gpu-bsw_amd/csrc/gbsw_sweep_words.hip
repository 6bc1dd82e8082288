// gbsw_sweep_words.hip -- sweep kernels with four pairs per wave: 16-bit profile.
#include "gbsw_sweep.hpp"

namespace gbsw {

const void* sweep_kernel_words(int kind, int)
{
    return (kind & kWideLanes) ? (const void*)&k_sweep<Sweep16, 16, kProfWords, true> : (const void*)&k_sweep<Sweep16, 16, kProfWords, false>;
}

} // namespace gbsw
