// One-launch Bluestein kernel, float.
#include "kblue.hpp"

namespace afft {

const void* mix_blue_kernel_c64() { return (const void*)&k_mix_blue<float, false>; }

}  // namespace afft
