// Runtime-size mixed-radix kernels, complex64, column layouts.
#include "kmix.hpp"

namespace afft {

const void* mix_kernel_c64_cols(int var, int dir) {
    if (var == VAR_COL) return dir < 0 ? (const void*)&k_mix<float, VAR_COL, -1> : (const void*)&k_mix<float, VAR_COL, 1>;
    return dir < 0 ? (const void*)&k_mix<float, VAR_4A, -1> : (const void*)&k_mix<float, VAR_4A, 1>;
}

}  // namespace afft
