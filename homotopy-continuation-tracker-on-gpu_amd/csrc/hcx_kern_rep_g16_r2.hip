// Latency tracker kernel instances (FP64, 2 replicas per path): generic, NMAX = 16.
#include "hcx_kernel.hpp"

namespace hcx {

KernelFn kernel_rep_g16_r2(int deg) {
  switch (deg) {
    case 2: return track_kernel_rep<16, 2, false, 2>;
    case 3: return track_kernel_rep<16, 3, false, 2>;
    case 4: return track_kernel_rep<16, 4, false, 2>;
    case 6: return track_kernel_rep<16, 6, false, 2>;
    default: return nullptr;
  }
}

}  // namespace hcx
