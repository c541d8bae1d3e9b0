// Latency tracker kernel instances (FP64) of 2 or 4 replicas per path, columns
// dealt out: size-specialised, n = G in {3, 4, 5, 6, 8, 9, 10, 12, 16}.
#include "hcx_kernel.hpp"

namespace hcx {

namespace {
template <int N>
KernelFn pick(int deg, int R) {
  if (R == 2) return deg <= 2 ? track_kernel_rep<N, 2, true, 2, true> : track_kernel_rep<N, 3, true, 2, true>;
  return deg <= 2 ? track_kernel_rep<N, 2, true, 4, true> : track_kernel_rep<N, 3, true, 4, true>;
}
}  // namespace

KernelFn kernel_deal_x(int n, int deg, int R) {
  if (deg > 3 || (R != 2 && R != 4)) return nullptr;
  switch (n) {
    case 3: return pick<3>(deg, R);
    case 4: return pick<4>(deg, R);
    case 5: return pick<5>(deg, R);
    case 6: return pick<6>(deg, R);
    case 8: return pick<8>(deg, R);
    case 9: return pick<9>(deg, R);
    case 10: return pick<10>(deg, R);
    case 12: return pick<12>(deg, R);
    case 16: return pick<16>(deg, R);
    default: return nullptr;
  }
}

}  // namespace hcx
