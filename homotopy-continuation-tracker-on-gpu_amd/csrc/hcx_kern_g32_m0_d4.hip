// Generic tracker kernel instance: NMAX = 32, terms of up to 4 variable factors, FP64 mode.
#include "hcx_kernel.hpp"

namespace hcx {

KernelFn kernel_g32_m0_d4() { return track_kernel<32, 4, 0, false>; }

}  // namespace hcx
