// Runtime-size mixed-radix real-row kernels, float.
#include "kmix.hpp"

namespace afft {

const void* mix_real_kernel_c64(int dir) {
    return dir < 0 ? (const void*)&k_mix_real<float, -1> : (const void*)&k_mix_real<float, 1>;
}

}  // namespace afft
