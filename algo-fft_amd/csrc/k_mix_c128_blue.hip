// One-launch Bluestein kernel, double.
#include "kblue.hpp"

namespace afft {

const void* mix_blue_kernel_c128() { return (const void*)&k_mix_blue<double, false>; }

}  // namespace afft
