// Runtime-size mixed-radix real-row kernels, double.
#include "kmix.hpp"

namespace afft {

const void* mix_real_kernel_c128(int dir) {
    return dir < 0 ? (const void*)&k_mix_real<double, -1> : (const void*)&k_mix_real<double, 1>;
}

}  // namespace afft
