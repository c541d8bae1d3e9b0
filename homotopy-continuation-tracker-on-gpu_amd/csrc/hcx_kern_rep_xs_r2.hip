// Latency tracker kernel instances (FP64, 2 replicas per path): size-specialised,
// n = G in {3, 4, 5, 6}, n = 4, 5 up to degree 4.
#include "hcx_kernel.hpp"

namespace hcx {

KernelFn kernel_rep_xs_r2(int n, int deg) {
  if (deg > 4 || (deg == 4 && n != 4 && n != 5)) return nullptr;
  const bool d2 = deg <= 2;
  switch (n) {
    case 3: return d2 ? track_kernel_rep<3, 2, true, 2> : track_kernel_rep<3, 3, true, 2>;
    case 4:
      if (deg == 4) return track_kernel_rep<4, 4, true, 2>;
      return d2 ? track_kernel_rep<4, 2, true, 2> : track_kernel_rep<4, 3, true, 2>;
    case 5:
      if (deg == 4) return track_kernel_rep<5, 4, true, 2>;
      return d2 ? track_kernel_rep<5, 2, true, 2> : track_kernel_rep<5, 3, true, 2>;
    case 6: return d2 ? track_kernel_rep<6, 2, true, 2> : track_kernel_rep<6, 3, true, 2>;
    default: return nullptr;
  }
}

}  // namespace hcx
