// Latency tracker kernel instances (FP64, the launch's number of replicas): generic, NMAX = 8.
#include "hcx_kernel.hpp"

namespace hcx {

KernelFn kernel_rep_g8_r1(int deg) {
  switch (deg) {
    case 2: return track_kernel_rep<8, 2, false, 1>;
    case 3: return track_kernel_rep<8, 3, false, 1>;
    case 4: return track_kernel_rep<8, 4, false, 1>;
    case 6: return track_kernel_rep<8, 6, false, 1>;
    default: return nullptr;
  }
}

}  // namespace hcx
