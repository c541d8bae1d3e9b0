// Generic tracker kernel instance: NMAX = 16, terms of up to 4 variable factors, FP64 mode.
#include "hcx_kernel.hpp"

namespace hcx {

KernelFn kernel_g16_m0_d4() { return track_kernel<16, 4, 0, false>; }

}  // namespace hcx
