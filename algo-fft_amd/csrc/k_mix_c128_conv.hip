// One-launch convolution kernels, double.
#include "kconv.hpp"

namespace afft {

const void* mix_conv_kernel_c128(bool real) {
    return real ? (const void*)&k_mix_conv<double, true> : (const void*)&k_mix_conv<double, false>;
}

}  // namespace afft
