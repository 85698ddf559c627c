// Runtime-size mixed-radix kernels, complex128, row layouts.
#include "kmix.hpp"

namespace afft {

const void* mix_kernel_c128_rows(int var, int dir) {
    if (var == VAR_ROW) return dir < 0 ? (const void*)&k_mix<double, VAR_ROW, -1> : (const void*)&k_mix<double, VAR_ROW, 1>;
    return dir < 0 ? (const void*)&k_mix<double, VAR_4B, -1> : (const void*)&k_mix<double, VAR_4B, 1>;
}

}  // namespace afft
