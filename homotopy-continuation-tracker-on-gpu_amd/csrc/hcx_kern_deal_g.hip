// Latency tracker kernel instances (FP64) of 2 or 4 replicas per path, columns
// dealt out: generic, NMAX = 8 and 16.
#include "hcx_kernel.hpp"

namespace hcx {

KernelFn kernel_deal_g(int nmax, int deg, int R) {
  if (deg > 3 || (R != 2 && R != 4)) return nullptr;
  const bool d2 = deg <= 2;
  if (nmax == 8) {
    if (R == 2) return d2 ? track_kernel_rep<8, 2, false, 2, true> : track_kernel_rep<8, 3, false, 2, true>;
    return d2 ? track_kernel_rep<8, 2, false, 4, true> : track_kernel_rep<8, 3, false, 4, true>;
  }
  if (nmax == 16) {
    if (R == 2) return d2 ? track_kernel_rep<16, 2, false, 2, true> : track_kernel_rep<16, 3, false, 2, true>;
    return d2 ? track_kernel_rep<16, 2, false, 4, true> : track_kernel_rep<16, 3, false, 4, true>;
  }
  return nullptr;
}

}  // namespace hcx
