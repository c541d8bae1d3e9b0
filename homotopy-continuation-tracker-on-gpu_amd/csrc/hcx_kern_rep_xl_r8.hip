// Latency tracker kernel instances (FP64, 8 replicas per path): size-specialised,
// n = G = 8.
#include "hcx_kernel.hpp"

namespace hcx {

KernelFn kernel_rep_xl_r8(int n, int deg) {
  const bool d2 = deg <= 2;
  if (deg > 3) return nullptr;
  switch (n) {
    case 8: return d2 ? track_kernel_rep<8, 2, true, 8> : track_kernel_rep<8, 3, true, 8>;
    default: return nullptr;
  }
}

}  // namespace hcx
