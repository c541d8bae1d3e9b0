// Generic tracker kernel instance: NMAX = 8, terms of up to 4 variable factors, FP64 mode.
#include "hcx_kernel.hpp"

namespace hcx {

KernelFn kernel_g8_m0_d4() { return track_kernel<8, 4, 0, false>; }

}  // namespace hcx
