// One-launch convolution kernels, float.
#include "kconv.hpp"

namespace afft {

const void* mix_conv_kernel_c64(bool real) {
    return real ? (const void*)&k_mix_conv<float, true> : (const void*)&k_mix_conv<float, false>;
}

}  // namespace afft
