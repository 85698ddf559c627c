// Runtime-size mixed-radix kernels, complex128, column layouts.
#include "kmix.hpp"

namespace afft {

const void* mix_kernel_c128_cols(int var, int dir) {
    if (var == VAR_COL) return dir < 0 ? (const void*)&k_mix<double, VAR_COL, -1> : (const void*)&k_mix<double, VAR_COL, 1>;
    return dir < 0 ? (const void*)&k_mix<double, VAR_4A, -1> : (const void*)&k_mix<double, VAR_4A, 1>;
}

}  // namespace afft
