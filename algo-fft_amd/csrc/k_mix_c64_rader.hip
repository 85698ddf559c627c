// One-launch Rader kernel, float.
#include "kblue.hpp"

namespace afft {

const void* mix_rader_kernel_c64() { return (const void*)&k_mix_blue<float, true>; }

}  // namespace afft
