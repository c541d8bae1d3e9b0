// Latency tracker kernel instances (FP64, 2 replicas per path): generic, NMAX = 32.
#include "hcx_kernel.hpp"

namespace hcx {

KernelFn kernel_rep_g32_r2(int deg) {
  switch (deg) {
    case 2: return track_kernel_rep<32, 2, false, 2>;
    case 3: return track_kernel_rep<32, 3, false, 2>;
    case 4: return track_kernel_rep<32, 4, false, 2>;
    case 6: return track_kernel_rep<32, 6, false, 2>;
    default: return nullptr;
  }
}

}  // namespace hcx
