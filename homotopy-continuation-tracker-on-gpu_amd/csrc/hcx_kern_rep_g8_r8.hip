// Latency tracker kernel instances (FP64, 8 replicas per path): generic, NMAX = 8.
#include "hcx_kernel.hpp"

namespace hcx {

KernelFn kernel_rep_g8_r8(int deg) {
  switch (deg) {
    case 2: return track_kernel_rep<8, 2, false, 8>;
    case 3: return track_kernel_rep<8, 3, false, 8>;
    case 4: return track_kernel_rep<8, 4, false, 8>;
    case 6: return track_kernel_rep<8, 6, false, 8>;
    default: return nullptr;
  }
}

}  // namespace hcx
