// Strided copy and stand-alone real recombination kernels.
#include "kernels.hpp"

namespace afft {

const void* copy_kernel(int prec) {
    return prec == 0 ? (const void*)&k_copy<float> : (const void*)&k_copy<double>;
}

const void* rpost_kernel(int prec, int dir) {
    if (prec == 0) return dir < 0 ? (const void*)&k_rpost<float, -1> : (const void*)&k_rpost<float, 1>;
    return dir < 0 ? (const void*)&k_rpost<double, -1> : (const void*)&k_rpost<double, 1>;
}

const void* mix_kernel_c64_rows(int var, int dir);
const void* mix_kernel_c64_cols(int var, int dir);
const void* mix_kernel_c128_rows(int var, int dir);
const void* mix_kernel_c128_cols(int var, int dir);

// k_mix of one precision, variant and direction.
const void* mix_kernel(int prec, int var, int dir) {
    const bool cols = var == VAR_COL || var == VAR_4A;
    if (prec == 0) return cols ? mix_kernel_c64_cols(var, dir) : mix_kernel_c64_rows(var, dir);
    return cols ? mix_kernel_c128_cols(var, dir) : mix_kernel_c128_rows(var, dir);
}

const void* mix_real_kernel_c64(int dir);
const void* mix_real_kernel_c128(int dir);

const void* mix_real_kernel(int prec, int dir) { return prec ? mix_real_kernel_c128(dir) : mix_real_kernel_c64(dir); }

}  // namespace afft
