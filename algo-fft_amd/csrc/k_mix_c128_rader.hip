// One-launch Rader kernel, double.
#include "kblue.hpp"

namespace afft {

const void* mix_rader_kernel_c128() { return (const void*)&k_mix_blue<double, true>; }

}  // namespace afft
