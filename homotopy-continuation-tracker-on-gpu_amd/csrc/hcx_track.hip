// gfx950 path tracker: persistent lane-group kernel, launchers and the
// tracking half of the C-ABI.
//
// Method (per path) restates the reference kernel loop
// GPU-HC/magmaHC/gpu-kernels/kernel_HC_Solver_generalized_3views_4pts.cu:115-260:
// end-zone clamp (:121-131), "loopy" RK4 predictor (:139-183), Newton
// corrector with |dx|^2 < tol |x|^2 success and |x|^2 > 1e14 infinity tests
// (:189-225), halving / doubling step control (:230-249), outputs (:256-264).
// Table semantics follow dev-eval-indxing-generalized_3views_4pts.cuh:34-120,
// the solve follows dev-cgesv-batched-small.cuh:38-107 (cabs1 partial pivoting,
// first maximum in current row order, elimination with the pivot's reciprocal).
//
// Work decomposition (MI355X-first): a wave64 holds floor(64/G) lane groups;
// each group tracks one path at a time, lane gl < n owns equation gl.  Groups
// refill from a device work counter as soon as their path ends, so a wave
// never idles on its slowest path.  Paths of several problem types
// ("segments") share one launch; a wave works a segment until its queue is
// empty and then steals from the others.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <vector>

#include "hcx_internal.hpp"
#include "hcx_kernel.hpp"

namespace hcx {

using dev::cx;
using dev::cmk;

struct OutPack {
  SegOut out[kMaxSeg];
};

// Launch set-up on the device (graph-safe, no memset): path queues, lengths of
// the re-track lists, per-instance remaining-path counters, output
// descriptors, start stamp.
__global__ void init_kernel(const Launch LN, const OutPack OP, unsigned long long* batch_start) {
  const int s = blockIdx.y;
  if (s >= LN.nseg) return;
  const Seg& S = LN.seg[s];
  const SegOut& O = OP.out[s];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) {
    *S.counter = 0u;
    if (S.plist_count) S.plist_count[0] = S.plist_count[1] = 0u;
    *const_cast<SegOut*>(S.out) = O;
  }
  if (O.inst_left && i < S.I) O.inst_left[i] = S.K;
  if (batch_start && s == 0 && i == 0) *batch_start = wall_clock64();
}

// Parameter-affine P2C on the device: c_j(p) = A[j][0] + sum_q A[j][1+q] p_q
// for p0 and p1 of each instance, written as the M = 1 coefficient tables
// Hx[i][j] = {c(p0), c(p1) - c(p0)}, Ht[i][j] = {c(p1) - c(p0)}, entry C = {1, 0}
// (the role of Data_Reader::Construct_Coeffs_From_Params, Data_Reader.cpp:59-89).
__global__ void p2c_affine_kernel(const double2* __restrict__ A, int C, int k, const double2* __restrict__ p0,
                                  int p0_stride, const double2* __restrict__ p1, int I, double2* __restrict__ hx,
                                  double2* __restrict__ ht) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = blockIdx.y;
  if (j > C || i >= I) return;
  double2* hxi = hx + ((size_t)i * (C + 1) + j) * 2;
  double2* hti = ht + ((size_t)i * (C + 1) + j);
  if (j == C) {
    hxi[0] = make_double2(1.0, 0.0);
    hxi[1] = make_double2(0.0, 0.0);
    hti[0] = make_double2(0.0, 0.0);
    return;
  }
  const double2* a = A + (size_t)j * (1 + k);
  const double2* q0 = p0 + (size_t)i * p0_stride;
  const double2* q1 = p1 + (size_t)i * k;
  double r0 = a[0].x, i0 = a[0].y, r1 = a[0].x, i1 = a[0].y;
  for (int q = 0; q < k; ++q) {
    const double2 c = a[1 + q], u = q0[q], v = q1[q];
    r0 += c.x * u.x - c.y * u.y;
    i0 += c.x * u.y + c.y * u.x;
    r1 += c.x * v.x - c.y * v.y;
    i1 += c.x * v.y + c.y * v.x;
  }
  hxi[0] = make_double2(r0, i0);
  hxi[1] = make_double2(r1 - r0, i1 - i0);
  hti[0] = make_double2(r1 - r0, i1 - i0);
}

// Parameter-polynomial P2C on the device: for instance i and coefficient j,
// c_j(p(t)) with p(t) = p0 + t (p1 - p0) and
// c_j(p) = sum_u scalar[j][u] prod_d p[params[j][u][d]] (p[k] = 1) as its
// t^0..t^M coefficients Hx[i][j][0..M] and those of dc_j/dt, Ht[i][j][0..M-1]
// (the role of the generated p2c-<p>.h, Data_Reader.cpp:59-89, with the
// coefficient-polynomial layout of createUnivPoly4Coeffs.m; entry C = {1, 0..}).
// Each term is a product of linear factors (q_a + t d_a), expanded by
// repeated polynomial multiplication.
constexpr int kMaxOrderT = 8;

__global__ void p2c_poly_kernel(const double2* __restrict__ scal, const int* __restrict__ prm, int C, int T, int D,
                                int k, int M, const double2* __restrict__ p0, int p0_stride,
                                const double2* __restrict__ p1, int I, double2* __restrict__ hx,
                                double2* __restrict__ ht) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = blockIdx.y;
  if (j > C || i >= I) return;
  double2* hxi = hx + ((size_t)i * (C + 1) + j) * (M + 1);
  double2* hti = ht + ((size_t)i * (C + 1) + j) * M;
  double cr[kMaxOrderT + 1], ci[kMaxOrderT + 1];
#pragma unroll
  for (int m = 0; m <= kMaxOrderT; ++m) cr[m] = ci[m] = 0.0;
  if (j == C) {
    cr[0] = 1.0;
  } else {
    const double2* q0 = p0 + (size_t)i * p0_stride;
    const double2* q1 = p1 + (size_t)i * k;
    for (int u = 0; u < T; ++u) {
      const double2 sc = scal[(size_t)j * T + u];
      if (sc.x == 0.0 && sc.y == 0.0) continue;
      double tr[kMaxOrderT + 1], ti[kMaxOrderT + 1];
#pragma unroll
      for (int m = 0; m <= kMaxOrderT; ++m) tr[m] = ti[m] = 0.0;
      tr[0] = sc.x;
      ti[0] = sc.y;
      int deg = 0;
      for (int d = 0; d < D; ++d) {
        const int a = prm[((size_t)j * T + u) * D + d];
        if (a >= k) continue;  // the constant-1 padding factor
        const double2 qa = q0[a], pa = q1[a];
        const double dr = pa.x - qa.x, di = pa.y - qa.y;
        // (tr, ti) *= (qa + t d): new[m] = old[m] qa + old[m-1] d
#pragma unroll
        for (int m = kMaxOrderT; m >= 0; --m) {
          if (m > deg + 1) continue;
          double nr = tr[m] * qa.x - ti[m] * qa.y, ni = tr[m] * qa.y + ti[m] * qa.x;
          if (m > 0) {
            nr += tr[m - 1] * dr - ti[m - 1] * di;
            ni += tr[m - 1] * di + ti[m - 1] * dr;
          }
          tr[m] = nr;
          ti[m] = ni;
        }
        ++deg;
      }
#pragma unroll
      for (int m = 0; m <= kMaxOrderT; ++m) {
        cr[m] += tr[m];
        ci[m] += ti[m];
      }
    }
  }
#pragma unroll
  for (int m = 0; m <= kMaxOrderT; ++m) {
    if (m <= M) hxi[m] = make_double2(cr[m], ci[m]);
    if (m < M) hti[m] = make_double2((m + 1) * cr[m + 1], (m + 1) * ci[m + 1]);
  }
}

__device__ __forceinline__ bool same_root(const double2* a, const double2* b, int n, double tol) {
  for (int v = 0; v < n; ++v)
    if (!(fabs(a[v].x - b[v].x) < tol && fabs(a[v].y - b[v].y) < tol)) return false;
  return true;
}

// Solution collection on the device, one block per instance
// (Evaluations.cpp:88-176).  Counts [tracked, infinity, refined, real,
// unique, unique_ref, real_ref]:
//  * unique: first occurrence of a refined root among the refined roots;
//  * real_ref: tracked paths carrying HCX_FLAG_REAL_REF, the reference's real
//    test on the tracked root (Evaluate_GPUHC_Sols, :88-110);
//  * unique_ref: Find_Unique_Sols (:127-176).  Its Skip set is always the
//    Duplicate set of the last examined path that had one (bstar), so the
//    sequential pass needs, per path, only "has a later path (any outcome)
//    with the same root" and a comparison with bstar.
// The pair comparisons run in parallel over the block (thread per first
// index, roots staged in LDS when they fit) into LDS bit sets; one thread
// then runs the short sequential pass.  Dynamic LDS: 4 bit sets of
// ceil(K / 32) words, then K * n roots when stage_roots is set.
__global__ void collect_kernel(int n, int K, const double2* __restrict__ roots, uint32_t* __restrict__ flags,
                               double tol, unsigned long long* __restrict__ counts, int stage_roots) {
  extern __shared__ __align__(16) unsigned int bits[];
  const int words = (K + 31) / 32;
  unsigned int* later = bits;                // a later path (any outcome) has the same root
  unsigned int* tracked = bits + words;      // tracked ("converged")
  unsigned int* dupref = bits + 2 * words;   // refined with an earlier refined duplicate
  unsigned int* uref = bits + 3 * words;     // counted by the unique_ref pass
  double2* sroots = reinterpret_cast<double2*>(bits + ((4 * words + 3) & ~3));
  const int inst = blockIdx.x;
  const size_t base = (size_t)inst * K;
  for (int w = threadIdx.x; w < 4 * words; w += blockDim.x) bits[w] = 0u;
  const double2* x = roots + base * n;
  if (stage_roots) {
    for (int q = threadIdx.x; q < K * n; q += blockDim.x) sroots[q] = x[q];
    x = sroots;
  }
  __syncthreads();
  unsigned long long c_tr = 0, c_inf = 0, c_ref = 0, c_real = 0, c_rref = 0;
  for (int i = threadIdx.x; i < K; i += blockDim.x) {
    const uint32_t fi = flags[base + i];
    if (fi & HCX_FLAG_TRACKED) {
      ++c_tr;
      atomicOr(&tracked[i >> 5], 1u << (i & 31));
      if (fi & HCX_FLAG_REAL_REF) ++c_rref;
    }
    c_inf += (fi & HCX_FLAG_INFINITY) ? 1 : 0;
    const bool ri = (fi & HCX_FLAG_REFINED) != 0;
    if (ri) {
      ++c_ref;
      c_real += (fi & HCX_FLAG_REAL) ? 1 : 0;
    }
    bool lat = false;
    for (int j = i + 1; j < K; ++j) {
      if (!same_root(x + (size_t)i * n, x + (size_t)j * n, n, tol)) continue;
      lat = true;
      if (ri && (flags[base + j] & HCX_FLAG_REFINED)) atomicOr(&dupref[j >> 5], 1u << (j & 31));
    }
    if (lat) atomicOr(&later[i >> 5], 1u << (i & 31));
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long c_uref = 0;
    int bstar = -1;
    for (int bs = 0; bs < K; ++bs) {
      if (!((tracked[bs >> 5] >> (bs & 31)) & 1u)) continue;
      if (bstar >= 0 && same_root(x + (size_t)bs * n, x + (size_t)bstar * n, n, tol)) continue;
      if ((later[bs >> 5] >> (bs & 31)) & 1u) {
        bstar = bs;
      } else {
        uref[bs >> 5] |= 1u << (bs & 31);
        ++c_uref;
      }
    }
    atomicAdd(&counts[5], c_uref);
  }
  __syncthreads();
  unsigned long long c_uni = 0;
  for (int j = threadIdx.x; j < K; j += blockDim.x) {
    uint32_t f = flags[base + j] & ~(HCX_FLAG_UNIQUE | HCX_FLAG_UNIQUE_REF);
    if ((f & HCX_FLAG_REFINED) && !((dupref[j >> 5] >> (j & 31)) & 1u)) {
      f |= HCX_FLAG_UNIQUE;
      ++c_uni;
    }
    if ((uref[j >> 5] >> (j & 31)) & 1u) f |= HCX_FLAG_UNIQUE_REF;
    flags[base + j] = f;
  }
  atomicAdd(&counts[0], c_tr);
  atomicAdd(&counts[1], c_inf);
  atomicAdd(&counts[2], c_ref);
  atomicAdd(&counts[3], c_real);
  atomicAdd(&counts[4], c_uni);
  atomicAdd(&counts[6], c_rref);
}

// Lists the paths that the FP64 pass of a mixed-precision launch re-tracks from
// t = 0 (grid.x: instances, grid.y: segments).  Round 0: every path without a
// refined root (precision escalation) and, with dups, every refined path whose
// root equals another refined root of its instance (|dRe|, |dIm| < tol in every
// coordinate): a path that jumped onto another path's root shares that root.
// Round 1, when the paths of round 0 have their FP64 roots: every path still of
// mixed precision whose root equals one of those.  Also prepares the segment's
// path queue and output descriptor for the launch that follows (a re-tracked path
// does not count its instance's paths down again).
// Round 1 reads the flags only where no path of the instance was re-tracked.
__global__ void list_retrack_kernel(const Launch LN, double tol, int round, int dups) {
  const Seg& S = LN.seg[blockIdx.y];
  const int inst = blockIdx.x, n = S.n, K = S.K;
  if (inst == 0 && threadIdx.x == 0) {
    *S.counter = 0u;
    const_cast<SegOut*>(S.out)->inst_left = nullptr;
  }
  if (inst >= S.I) return;
  const size_t base = (size_t)inst * K;
  const uint32_t* const flags = S.out->flags + base;
  const double2* const roots = S.out->roots + base * n;
  // the roots compared with
  const uint32_t with = round == 0 ? HCX_FLAG_REFINED : HCX_FLAG_REFINED | HCX_FLAG_ESCALATED;
  if (round > 0) {
    __shared__ int any;
    if (threadIdx.x == 0) any = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < K; i += blockDim.x)
      if ((flags[i] & with) == with) any = 1;
    __syncthreads();
    if (!any) return;
  }
  for (int j = threadIdx.x; j < K; j += blockDim.x) {
    const uint32_t fj = flags[j];
    if (fj & HCX_FLAG_ESCALATED) continue;
    bool list = !(fj & HCX_FLAG_REFINED);
    if (!list && dups) {
      const double2* xj = roots + (size_t)j * n;
      for (int i = 0; i < K && !list; ++i)
        list = i != j && (flags[i] & with) == with && same_root(roots + (size_t)i * n, xj, n, tol);
    }
    if (list) S.plist[atomicAdd(S.plist_count, 1u)] = (int)(base + j);
  }
}

__global__ void zero_u64_kernel(unsigned long long* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0ull;
}

// ------------------------------------------------------------ dispatch table
static const int kNmaxList[] = {8, 16, 32};
static const int kDegList[] = {2, 3, 4, 6};

static KernelFn pick_kernel(int nmax, int deg, int mode) {
  switch (nmax) {
    case 8: return mode == 0 ? kernel_g8_m0(deg) : kernel_g8_m1(deg);
    case 16: return mode == 0 ? kernel_g16_m0(deg) : kernel_g16_m1(deg);
    case 32: return mode == 0 ? kernel_g32_m0(deg) : kernel_g32_m1(deg);
    default: return nullptr;
  }
}

// The latency instance of R replicas with the columns dealt out (nullptr: none).
static KernelFn pick_deal(int nmax, int deg, bool exact, int R) {
  return exact ? kernel_deal_x(nmax, deg, R) : kernel_deal_g(nmax, deg, R);
}

// The latency instance of R replicas (nullptr: none).  Numbers of replicas
// that have no instance of their own run on R = 1's, which takes any.
static KernelFn pick_rep(int nmax, int deg, bool exact, int R) {
  if (exact) {
    if (deg > 4) return nullptr;
    deg = deg < 2 ? 2 : deg;
    if (nmax >= 3 && nmax <= 6) {
      switch (R) {
        case 2: return kernel_rep_xs_r2(nmax, deg);
        case 4: return kernel_rep_xs_r4(nmax, deg);
        case 8: return kernel_rep_xs_r8(nmax, deg);
        default: return kernel_rep_xs_r1(nmax, deg);
      }
    }
    if (nmax == 8 || nmax == 9 || nmax == 10 || nmax == 12 || nmax == 16) {
      switch (R) {
        case 2: return kernel_rep_xl_r2(nmax, deg);
        case 4: return kernel_rep_xl_r4(nmax, deg);
        case 8: return kernel_rep_xl_r8(nmax, deg);
        default: return kernel_rep_xl_r1(nmax, deg);
      }
    }
    return nullptr;
  }
  switch (nmax) {
    case 8:
      switch (R) {
        case 2: return kernel_rep_g8_r2(deg);
        case 4: return kernel_rep_g8_r4(deg);
        case 8: return kernel_rep_g8_r8(deg);
        default: return kernel_rep_g8_r1(deg);
      }
    case 16: return R == 4 ? kernel_rep_g16_r4(deg) : R == 2 ? kernel_rep_g16_r2(deg) : kernel_rep_g16_r1(deg);
    case 32: return R == 2 ? kernel_rep_g32_r2(deg) : kernel_rep_g32_r1(deg);
    default: return nullptr;
  }
}

static KernelFn pick_exact(int n, int deg, int mode) {
  // degree 4 (8-byte compact terms of four variables): n = 4, 5 in FP64 mode
  if (deg > 4 || (deg == 4 && mode != 0)) return nullptr;
  deg = deg < 2 ? 2 : deg;
  switch (n) {
    case 3: return mode == 0 ? kernel_x3_m0(deg) : kernel_x3_m1(deg);
    case 4: return mode == 0 ? kernel_x4_m0(deg) : kernel_x4_m1(deg);
    case 5: return mode == 0 ? kernel_x5_m0(deg) : kernel_x5_m1(deg);
    case 6: return mode == 0 ? kernel_x6_m0(deg) : kernel_x6_m1(deg);
    case 8: return mode == 0 ? kernel_x8_m0(deg) : kernel_x8_m1(deg);
    case 9: return mode == 0 ? kernel_x9_m0(deg) : kernel_x9_m1(deg);
    case 10: return mode == 0 ? kernel_x10_m0(deg) : kernel_x10_m1(deg);
    case 12: return mode == 0 ? kernel_x12_m0(deg) : kernel_x12_m1(deg);
    case 16: return mode == 0 ? kernel_x16_m0(deg) : kernel_x16_m1(deg);
    case 30: return mode == 0 ? kernel_x30_m0(deg) : kernel_x30_m1(deg);
    default: return nullptr;
  }
}

}  // namespace hcx

#include "hcx_problem.hpp"


namespace hcx {
namespace {

std::mutex g_mu;
unsigned long long* g_counts = nullptr;   // device [kNumCounts], hcx_collect's totals
int g_cu = 0;
constexpr int kNumCounts = 7;
static_assert(kSegSlots == kMaxSeg, "workspace blocks hold one counter slot per segment");

#define HIP_TRY(expr)                                                              \
  do {                                                                             \
    hipError_t e_ = (expr);                                                        \
    if (e_ != hipSuccess) {                                                        \
      set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
      return HCX_ERR_HIP;                                                          \
    }                                                                              \
  } while (0)

// Compute-unit count of the device (sizes persistent grids); allocates nothing.
hcx_status ensure_device_info() {
  std::lock_guard<std::mutex> lk(g_mu);
  if (g_cu > 0) return HCX_OK;
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  HIP_TRY(hipGetDeviceProperties(&prop, dev));
  g_cu = prop.multiProcessorCount;
  return HCX_OK;
}

// Device-memory policy of the workspace pool.
struct HipDev {
  void* alloc(size_t n) {
    void* p = nullptr;
    return hipMalloc(&p, n) == hipSuccess ? p : nullptr;
  }
  void release(void* p) { (void)hipFree(p); }
  bool sync(const void* s) { return hipStreamSynchronize((hipStream_t)s) == hipSuccess; }
  bool capturing(const void* s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing((hipStream_t)s, &st) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    return st == hipStreamCaptureStatusActive;
  }
};

// Per-stream launch workspaces; lives until the process ends (blocks that
// captured graphs refer to must outlive every graph).
WorkspacePool<HipDev>& pool() {
  static auto* p = new WorkspacePool<HipDev>(HipDev{}, sizeof(SegOut));
  return *p;
}

hcx_status ws_error(WsStatus w, const char* who) {
  switch (w) {
    case WsStatus::kOk: return HCX_OK;
    case WsStatus::kCaptureTooSmall:
      set_error("%s: the stream's launch workspace is too small and cannot grow during graph capture; "
                "run the same launch once on this stream before capturing it", who);
      return HCX_ERR_INVALID_ARG;
    case WsStatus::kOutOfMemory:
      set_error("%s: out of device memory for the launch workspace", who);
      return HCX_ERR_OUT_OF_MEMORY;
    default:
      set_error("%s: waiting for the stream before growing its workspace failed", who);
      return HCX_ERR_HIP;
  }
}

int round_up_idx(const int* list, int cnt, int v) {
  for (int i = 0; i < cnt; ++i)
    if (list[i] >= v) return i;
  return -1;
}

double f_term(int d) { return 6.0 * d + 4.0; }

// LAPACK Working Note 41 counts for one complex GETRF + GETRS with 1 RHS.
double f_lu(int n) { return (8.0 / 3.0) * n * n * n + 7.0 * n * n + (7.0 / 3.0) * n; }

hcx_status validate_opts(const hcx_track_opts* o) {
  if (!o) {
    set_error("options are NULL");
    return HCX_ERR_INVALID_ARG;
  }
  if (o->max_steps < 0 || o->max_corr < 1 || o->incr_steps < 1 || !(o->dt0 > 0) || !(o->end_zone >= 0) ||
      !(o->t_tol > 0) || o->refine_iters < 0 || (o->precision != HCX_PREC_FP64 && o->precision != HCX_PREC_MIXED) ||
      o->lanes_per_path < 0 || o->lanes_per_path > 64 || o->specialize < 0 || o->specialize > 1 ||
      o->waves_per_cu < -64 || o->waves_per_cu > 64 || o->replicas < 0 || o->replicas > 64 ||
      (o->replicas & (o->replicas - 1)) != 0) {
    set_error("invalid tracker options (max_steps=%d max_corr=%d incr=%d precision=%d lanes=%d)", o->max_steps,
              o->max_corr, o->incr_steps, o->precision, o->lanes_per_path);
    return HCX_ERR_INVALID_ARG;
  }
  return HCX_OK;
}

Opts to_opts(const hcx_track_opts* o) {
  Opts r;
  r.ez_enter = o->end_zone + 1e-7;
  r.ez_land = 1.0 - o->end_zone;
  r.max_steps = o->max_steps;
  r.max_corr = o->max_corr;
  r.incr = o->incr_steps;
  r.refine_iters = o->refine_iters;
  r.dt0 = o->dt0;
  r.t_tol = o->t_tol;
  r.dt_min = o->dt_min;
  r.corr_tol = o->corr_tol;
  r.inf_tol = o->inf_tol;
  r.refine_tol = o->refine_tol;
  r.real_tol = o->real_tol;
  r.real_ref_tol = o->real_ref_tol;
  r.newton32 = o->fp32_corrector ? 1 : 0;
  return r;
}

// Per-group LDS: the x / pivot-row slots (shared, FP64 capacity) and the
// constants 1 and 0, the pivot keys (instances without DPP groups) and the
// coefficient area of `slots` slots.  FP64: c(t), and dc/dt with M > 1 or
// dot_lds (with M = 1 dc/dt is constant and read from the instance's table in
// global memory); mixed: with M = 1 FP32 c + dc/dt overlaid by FP64 c.
// The region stride is an odd multiple of 16 bytes: the groups of a wave read
// the same offsets of their regions together (pivot-row broadcasts, x and
// coefficient gathers), and such a stride spreads them over distinct LDS banks
// (64 banks x 4 bytes) for 8- and 16-byte accesses.
int lds_group_bytes(int nmax, bool keys, int slots, int M, bool dot_lds = false) {
  const int per = (M > 1 || dot_lds) ? 32 : 16;
  const int b = 16 * (nmax + 2) + dev::key_bytes(keys) + slots * per;
  return (((b + 15) / 16) | 1) * 16;
}

// Form of the compact tables for terms of up to `deg` variables.
int compact_format(int deg) { return deg <= 2 ? 0 : (deg <= 4 ? 1 : 2); }

struct Plan {
  int nmax = 0, mode = 0;
  int deg = 2;       // term degree of the instance (generic: rounded up to its instance's)
  bool exact = false;
  bool latency = false;  // the latency instance, with its own compact tables
  int fmt = 0;       // the compact tables are those of degree <= 2 (0), 4 (1) or 6 (2)
  int tab_lds = 0;   // LDS bytes of the compact tables (instances that hold them there)
  size_t lds = 0;
  KernelFn fn = nullptr;
  bool keys() const { return latency || !(exact && is_pow2(exact_lanes(nmax))); }  // pivot keys in LDS
  int group_bytes(const hcx_problem* p, bool dot_lds = false) const {
    return lds_group_bytes(nmax, keys(), p->nslot, mode == 0 ? p->M : 1, dot_lds);
  }
};

// Largest compact table the size-specialised instances (up to n = 16; n = 30
// with quadratic terms) stage in
// LDS; a problem with larger tables runs on the generic instance.
constexpr int kMaxTabLds = 32 * 1024;
// The measure of that limit: the tables at their full width (every equation's
// and column's padded number of terms), 4 or 8 bytes a term; the compact
// streams drop the padding and take up to twice that for the terms of H.
long long table_bytes(const hcx_problem* p, bool t4) {
  return (((long long)p->hxT * p->n + p->htT_padded) * p->n * (t4 ? 4 : 8) + 15) / 16 * 16;
}
// LDS per workgroup on gfx950
constexpr int kMaxLdsBytes = 160 * 1024;

// Waves of `wave` bytes of LDS that fit a CU at once, blocks of any number of
// waves (at most cap) sharing `tab` bytes.
int resident_waves(size_t tab, size_t wave, int cap) {
  int w = 0;
  for (int wpb = 1; wpb <= cap; ++wpb) w = std::max(w, (int)(kMaxLdsBytes / (tab + wpb * wave)) * wpb);
  return std::min(w, cap);
}

// Replicas of a launch beyond those that split the term sums: the columns are
// dealt out instead, each summed whole, so the additions are those of one
// replica.
//
// Two replicas halve a path's step (0.45), and a launch of up to about two
// rounds of resident waves is as long as its longest paths, so they pay past
// the 8 waves that a CU holds: up to 16 per CU at up to 8 variables, 12 beyond
// or where pairs leave more lanes of the wave empty than single groups do.  Throughput instance -> R = 2, us,
// by waves at R = 1:
//   n = 3  1300: 1615 1576  2048: 1808 1662  3000: 1432 1611
//   n = 6  1300: 2055 2014  2048: 3272 3115  3000: 3253 3360
//   n = 8  1296: 2673 2398  2048: 3340 3016  4096: 4211 4346
//   n = 10 1302: 3432 3137  2048: 3833 4165
//   n = 9   609: 2779 2275  1300: 3000 2810  2049: 3324 3615
//   n = 12  589: 3415 3011  1306: 4165 4073  2048: 5053 5023  2996: 5620 6584
//
// Where LDS holds fewer waves of a CU than the registers (wide coefficient
// tables), R with the best rate of a full chip is taken at any number of
// waves: resident paths times the speed of their steps.  n = 16, 352
// coefficients: 24 paths in 6 waves -> 12 in 6 at R = 2, 4100 waves 14.3 -> 13.1 ms,
// 2050 10.4 -> 8.9; n = 10, 660 coefficients: 12 paths in 2 waves -> 7 in 7 at R = 4,
// 4096 waves 35.1 -> 30.5 ms, 598 11.6 -> 8.6.
template <class Region, class Waves>
int dealt_replicas(const Seg& S, const Plan& pl, int tab, const Region& region, const Waves& waves) {
  auto groups = [&](int R) { return 64 / (S.G * R); };
  int R = 1;
  if (2 * S.G <= 64 && waves(2) <= (groups(1) <= 2 * groups(2) && S.n <= 8 ? 16LL : 12LL) * g_cu) R = 2;
  const int cap = 4 * waves_per_simd(pl.nmax, pl.exact), capr = 4 * waves_per_simd(pl.nmax, false);
  const int w1 = resident_waves((size_t)pl.tab_lds, (size_t)groups(1) * S.lds_group, cap);
  if (w1 < cap) {
    const double speed[] = {1.0, 2.2, 2.9};
    double best = groups(1) * w1;
    for (int i = 1; i < 3 && (S.G << i) <= 64; ++i) {
      const double rate = speed[i] * groups(1 << i) *
                          resident_waves((size_t)tab, (size_t)groups(1 << i) * region(1 << i), capr);
      if (rate > best) {
        best = rate;
        R = std::max(R, 1 << i);
      }
    }
  }
  return R;
}

// Kernel instance for a launch: the size-specialised one when every segment
// has the same n, runs its lanes per path (G = exact_lanes(n)) and fits
// DEG <= 3 (and, for
// n <= 16, has compact tables of at most kMaxTabLds bytes); the multi-size
// instance when the segments' sizes differ but all are in {3, 5, 6, 9, 12}
// with G = n, quadratic terms and compact tables; otherwise the generic
// instance with the smallest NMAX >= max n.
hcx_status choose_kernel(int nseg, const hcx_problem* const* probs, const int* Gs, int max_deg, int mode,
                         int specialize, Plan& pl) {
  pl.mode = mode;
  pl.tab_lds = 0;
  int max_n = 1, tab = 0;
  bool same = true, tab_ok = true, in_set = true;
  const bool t4 = max_deg <= 2;
  pl.fmt = compact_format(max_deg);
  for (int s = 0; s < nseg; ++s) {
    const int n = probs[s]->n;
    max_n = std::max(max_n, n);
    same = same && n == probs[0]->n && Gs[s] == exact_lanes(n);
    in_set = in_set && (n == 3 || n == 5 || n == 6 || n == 9 || n == 12) && Gs[s] == n;
    const auto& c = probs[s]->ctab[pl.fmt];
    tab_ok = tab_ok && c.d && table_bytes(probs[s], t4) <= kMaxTabLds;
    tab = std::max(tab, c.words * 4);
  }
  if (specialize && !same && in_set && tab_ok && max_deg <= 2) {
    pl.fn = mode == 0 ? kernel_set_m0() : kernel_set_m1();
    pl.nmax = max_n;
    pl.deg = 2;
    pl.exact = true;
    pl.tab_lds = tab;
    return HCX_OK;
  }
  const int n0 = probs[0]->n;
  // n = 30 holds the tables in LDS only with quadratic terms (4-byte records)
  if (specialize && same && (tab_ok || (n0 > 16 && !t4))) {
    KernelFn fn = pick_exact(n0, max_deg, mode);
    if (fn) {
      pl.fn = fn;
      pl.nmax = n0;
      pl.deg = max_deg;
      pl.exact = true;
      pl.tab_lds = (n0 <= 16 || t4) ? tab : 0;
      size_t lds = 0;
      for (int s = 0; s < nseg; ++s)
        lds = std::max(lds, (size_t)(64 / Gs[s]) * (size_t)pl.group_bytes(probs[s]) + (size_t)pl.tab_lds);
      if (lds <= (size_t)kMaxLdsBytes) return HCX_OK;
      pl.tab_lds = 0;
    }
  }
  const int ni = round_up_idx(kNmaxList, 3, max_n);
  int di = round_up_idx(kDegList, 4, max_deg);
  if (ni < 0 || di < 0) {
    set_error("unsupported sizes: n=%d (max %d), degree=%d (max 6)", max_n, kMaxN, max_deg);
    return HCX_ERR_UNSUPPORTED;
  }
  // terms of degree 3 or 4 with scalars beyond their compact form
  if (di >= 0 && nseg == 1 && pl.fmt == 1 && !probs[0]->ctab[1].d && probs[0]->ctab[2].d) {
    pl.fmt = 2;
    di = 3;
  }
  pl.fn = pick_kernel(kNmaxList[ni], kDegList[di], mode);
  pl.nmax = kNmaxList[ni];
  pl.deg = kDegList[di];
  pl.exact = false;
  if (nseg == 1 && pl.fn) {
    // a generic instance reads the compact streams from LDS where they take at
    // most 64 KiB and leave half the waves that a CU holds without them (its
    // registers allow one per SIMD for NMAX 32, else two): the records in
    // global memory cost more than half the waves.  1024 waves, ms, global -> LDS:
    // n = 7, degree 4, mixed (7 -> 6 waves) 19.3 -> 9.0; n = 18, 1080 coefficients (3 -> 2)
    // 37.8 -> 20.4; n = 28, 1680 coefficients (3 -> 2) 49.4 -> 29.1.
    const auto& c = probs[0]->ctab[pl.fmt];
    const size_t wave = (size_t)(64 / Gs[0]) * (size_t)pl.group_bytes(probs[0]), tb = (size_t)c.words * 4;
    const int cap = pl.nmax == 32 ? 4 : 8;
    if (c.d && tb <= 65536 && 2 * resident_waves(tb, wave, cap) >= resident_waves(0, wave, cap)) {
      pl.tab_lds = (int)tb;
    }
  }
  if (!pl.fn) {
    set_error("no kernel instance for n=%d degree=%d mode=%d", max_n, max_deg, mode);
    return HCX_ERR_UNSUPPORTED;
  }
  return HCX_OK;
}

// The tables of a segment in the form that the plan's kernel reads.
void seg_tables(Seg& S, const hcx_problem* p, const Plan& pl) {
  S.lds_group = pl.group_bytes(p);
  S.cslot = p->d_cslot;
  S.nslot = p->nslot;
  const auto& c = (pl.latency ? p->ltab : p->ctab)[pl.fmt];
  S.hx = p->d_hx;
  S.ht = p->d_ht;
  S.ht_ci = p->d_ht_ci;
  S.htT = p->htT;
  S.htS = p->htS;
  S.hx_recs = p->hx_recs;
  S.max_terms = p->max_terms;
  std::memcpy(S.colc, p->colc, sizeof(S.colc));
  S.hx_cnt = p->colc_fits ? nullptr : p->d_hx_cnt;
  S.ctab = pl.tab_lds > 0 ? c.d : nullptr;
  S.tab_words = c.words;
  S.tab_h = c.h;
  S.tab_slot = c.slot;
}

// Fills the segment-independent part of a Seg from a problem.
void seg_from_problem(Seg& S, SegOut& O, const hcx_problem* p, int G, const Plan& pl) {
  std::memset(&S, 0, sizeof(S));
  std::memset(&O, 0, sizeof(O));
  O.roots_stride = p->n;
  S.n = p->n;
  S.C = p->C;
  S.M = p->M;
  S.K = p->K;
  S.G = G;
  S.R = 1;
  seg_tables(S, p, pl);
  S.start = p->d_start;
  S.start_stride = p->n;
}

// Dynamic LDS bytes of a launch: the tables (when staged) and one region per
// full group of every wave of the block; the lanes of a partial group share
// their wave's region 0 and never write LDS.
size_t plan_lds(const Launch& LN, const Plan& pl) {
  size_t lds = 0;
  for (int s = 0; s < LN.nseg; ++s) {
    const Seg& S = LN.seg[s];
    const int groups = 64 / (S.G * S.R);
    lds = std::max(lds, (size_t)std::max(LN.wpb, 1) * (size_t)groups * (size_t)S.lds_group);
  }
  return lds + (size_t)pl.tab_lds;
}

hcx_status finish_plan(Launch& LN, Plan& pl) {
  if (LN.wpb < 1) LN.wpb = 1;
  const size_t lds = plan_lds(LN, pl);
  LN.tab_lds = pl.tab_lds;
  pl.lds = lds;
  if (lds > (size_t)kMaxLdsBytes) {
    set_error("launch needs %zu bytes of LDS per block (at most %d)", lds, kMaxLdsBytes);
    return HCX_ERR_UNSUPPORTED;
  }
  if (lds > 65536) {
    HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(pl.fn), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds));
  }
  return HCX_OK;
}

// Waves per block and blocks per CU of a persistent launch of `waves` waves.
// request: waves per CU; 0: as many as fit; negative: that many fewer (room for
// other solves in flight).  A request is never exceeded.
// Blocks of several waves only in one-segment launches whose instance holds
// the compact tables in LDS: the waves of a block share one copy of the
// tables, so they can leave room for more waves per CU.  The candidate with
// the most resident waves per CU within the request wins, the smaller block
// on ties; a launch takes no block that would leave a CU without one (blocks of
// 4 waves put 640 waves on 160 CUs).
// Against 1, 2 or 4 waves for any launch: n = 12, mixed, 21 KB per wave: 7 waves
// in place of 6, 150.3 -> 137.4 ms; 64 instances of n = 16 on 1280 waves: 5
// waves per CU in one block, 5.26 -> 4.84 ms.
hcx_status launch_density(Launch& LN, Plan& pl, long long waves, int request, int& blocks_per_cu) {
  const bool wide = LN.nseg == 1 && pl.tab_lds > 0;
  const int most = wide ? std::min(8, 4 * waves_per_simd(pl.nmax, pl.exact)) : 1;
  int resident[9] = {}, full = 1;
  for (int wpb = 1; wpb <= most && (wpb == 1 || waves >= (long long)wpb * g_cu); ++wpb) {
    LN.wpb = wpb;
    Plan q = pl;
    if (wpb > 1 && plan_lds(LN, q) > (size_t)kMaxLdsBytes) continue;
    hcx_status st = finish_plan(LN, q);
    if (st != HCX_OK) return st;
    int nb = 0;
    HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, reinterpret_cast<const void*>(pl.fn), 64 * wpb,
                                                         q.lds));
    resident[wpb] = nb * wpb;
    full = std::max(full, resident[wpb]);
  }
  const int limit = request > 0 ? request : std::max(full + request, 1);
  int best = -1;
  for (int wpb = 1; wpb <= std::min(most, limit); ++wpb) {
    const int w = std::min(resident[wpb], limit / wpb * wpb);
    if (w > best) {
      best = w;
      LN.wpb = wpb;
    }
  }
  blocks_per_cu = limit / LN.wpb;
  return finish_plan(LN, pl);
}

// Default lanes per path: those of the size-specialised instance (n, or 32
// for n = 30; several paths per wave, G need not divide 64), widened while
// the wave's groups would need more than 64 KiB of LDS (wide coefficient
// tables), so that at least two waves share a CU.
int default_lanes(int n, int C, int M) {
  const int ni = round_up_idx(kNmaxList, 3, n);
  const int lg = 16 * ((ni < 0 ? n : kNmaxList[ni]) + 1) + (C + 1) * (M > 1 ? 32 : 16) + 256;
  int G = exact_lanes(n);
  while (G < 64 && (size_t)(64 / G) * (size_t)lg > 65536) ++G;
  return G;
}

// Workspace entries a launch needs: instance counters when instance
// completion times are requested, the re-track list in mixed precision.
void ws_need(int nseg, hcx_problem* const* probs, const hcx_batch_desc* batches, const hcx_result_desc* results,
             const hcx_track_opts* o, long long& inst, long long& paths) {
  inst = paths = 0;
  for (int s = 0; s < nseg; ++s) {
    if (!probs[s] || batches[s].num_instances < 0) continue;
    const long long I = batches[s].num_instances;
    if (results[s].d_inst_done) inst += I;
    if (o && o->precision == HCX_PREC_MIXED) paths += I * probs[s]->K;
  }
}

// Carves the per-segment views of a block for the given launch.
void ws_carve(const WsBlock& b, int nseg, const hcx_batch_desc* batches, const hcx_result_desc* results,
              hcx_problem* const* probs, const hcx_track_opts* o, LaunchWork* work) {
  long long io = 0, po = 0;
  for (int s = 0; s < nseg; ++s) {
    work[s] = seg_work(b, s, io, po);
    const long long I = std::max(batches[s].num_instances, 0);
    if (results[s].d_inst_done) io += I;
    if (o->precision == HCX_PREC_MIXED && probs[s]) po += I * probs[s]->K;
  }
}

}  // namespace

LaunchWork seg_work(const WsBlock& b, int s, long long inst_off, long long path_off) {
  const WsLayout L = ws_layout(sizeof(SegOut), b.inst_cap, b.paths_cap);
  char* base = static_cast<char*>(b.base);
  LaunchWork w;
  w.counter = reinterpret_cast<unsigned int*>(base) + 64 * s;
  w.plist_count = w.counter + 32;
  w.out = reinterpret_cast<SegOut*>(base + L.out_off) + s;
  w.inst_left = reinterpret_cast<int*>(base + L.inst_off) + inst_off;
  w.plist = reinterpret_cast<int*>(base + L.plist_off) + path_off;
  w.inst_cap = b.inst_cap - inst_off;
  w.plist_cap = b.paths_cap - path_off;
  return w;
}

// ------------------------------------------------------------ static scratch
// Launch workspace of hcx_track_noalloc: a file-scope device array (each GPU
// holds its own copy until the process ends).  Host code never uses the
// array's name as an address: the device address comes from
// hipGetSymbolAddress, once per device, with that device current.
constexpr size_t kScratchBytes =
    ws_layout(sizeof(SegOut), HCX_NOALLOC_MAX_INSTANCES, HCX_NOALLOC_MAX_PATHS).bytes;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The current device's scratch as a workspace block.
hcx_status scratch_block(WsBlock& b) {
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("hcx_track_noalloc: device %d beyond the %d devices the scratch table covers", dev, kMaxDevices);
    return HCX_ERR_UNSUPPORTED;
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
      set_error("hcx_track_noalloc: hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
      return HCX_ERR_HIP;
    }
    g_scratch_ptr[dev] = p;
  }
  b.base = g_scratch_ptr[dev];
  b.inst_cap = HCX_NOALLOC_MAX_INSTANCES;
  b.paths_cap = HCX_NOALLOC_MAX_PATHS;
  b.pinned = true;
  return HCX_OK;
}
}  // namespace

// A launch on `stream` with that stream's pooled workspace.
hcx_status track_pooled(int nseg, hcx_problem* const* probs, const hcx_batch_desc* batches,
                        const hcx_result_desc* results, const hcx_track_opts* o, hipStream_t stream, int persistent,
                        unsigned long long* batch_start, const char* who) {
  if (nseg < 1 || nseg > kMaxSeg || !probs || !batches || !results || !o) {
    set_error("%s: need 1..%d segments with problems, batches, results and options", who, kMaxSeg);
    return HCX_ERR_INVALID_ARG;
  }
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  long long inst = 0, paths = 0;
  ws_need(nseg, probs, batches, results, o, inst, paths);
  WorkspacePool<HipDev>::Lease lease;
  hcx_status st = ws_error(pool().acquire(dev, stream, inst, paths, lease), who);
  if (st != HCX_OK) return st;
  LaunchWork work[kMaxSeg];
  ws_carve(lease.block(), nseg, batches, results, probs, o, work);
  return track_impl(nseg, probs, batches, results, o, stream, persistent, batch_start, work);
}

}  // namespace hcx

using namespace hcx;

extern "C" {

int hcx_device_count(void) {
  int c = 0;
  if (hipGetDeviceCount(&c) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return c;
}

hcx_status hcx_problem_create(const hcx_problem_desc* d, hcx_problem** out) {
  clear_error();
  if (!d || !out) {
    set_error("hcx_problem_create: null argument");
    return HCX_ERR_INVALID_ARG;
  }
  const int n = d->num_vars, C = d->num_coeffs, M = d->max_order_t;
  if (n < 1 || n > kMaxN || C < 1 || M < 1 || d->hx_terms < 1 || d->ht_terms < 1 || d->hx_parts < 3 ||
      d->ht_parts < 3 || d->hx_parts > 10 || d->ht_parts > 10 || !d->h_hx_idx || !d->h_ht_idx ||
      d->num_tracks < 1 || !d->h_start_sols || d->num_params < 0 ||
      (d->num_params > 0 && (!d->h_start_params || (!d->h_coeff_affine) == (!d->h_cmap_scalar)))) {
    set_error("hcx_problem_create: invalid descriptor (n=%d C=%d M=%d hx %dx%d ht %dx%d K=%d k=%d)", n, C, M,
              d->hx_terms, d->hx_parts, d->ht_terms, d->ht_parts, d->num_tracks, d->num_params);
    return HCX_ERR_INVALID_ARG;
  }
  if (d->h_cmap_scalar) {
    if (!d->h_cmap_params || d->cmap_terms < 1 || d->cmap_deg < 1 || d->cmap_deg > M || M > kMaxOrderT) {
      set_error("hcx_problem_create: invalid coefficient map (terms %d, degree %d, M %d; need 1 <= degree <= M <= %d)",
                d->cmap_terms, d->cmap_deg, M, kMaxOrderT);
      return HCX_ERR_INVALID_ARG;
    }
    const size_t np = (size_t)C * d->cmap_terms * d->cmap_deg;
    for (size_t q = 0; q < np; ++q)
      if (d->h_cmap_params[q] < 0 || d->h_cmap_params[q] > d->num_params) {
        set_error("hcx_problem_create: coefficient map parameter index %d out of range 0..%d", d->h_cmap_params[q],
                  d->num_params);
        return HCX_ERR_INVALID_ARG;
      }
  }
  if (hcx_device_count() < 1) {
    set_error("hcx_problem_create: no HIP device available");
    return HCX_ERR_NO_DEVICE;
  }
  hcx_status st = ensure_device_info();
  if (st != HCX_OK) return st;

  const int hxv = d->hx_parts - 2, htv = d->ht_parts - 2;
  // repack + validate tables: hx [var j][term][eq i], ht [term][eq i]
  std::vector<dev::Term> hx((size_t)n * d->hx_terms * n), ht((size_t)d->ht_terms * n);
  auto pack = [&](const int* rec, int nv, dev::Term& tm) -> bool {
    tm.s = rec[0];
    tm.c = rec[1];
    if (tm.c < 0 || tm.c > C) return false;
    uint32_t v03 = 0, v47 = 0;
    for (int q = 0; q < 8; ++q) {
      int v = q < nv ? rec[2 + q] : n;
      if (v < 0 || v > n) return false;
      if (q < 4) v03 |= (uint32_t)v << (8 * q);
      else v47 |= (uint32_t)v << (8 * (q - 4));
    }
    tm.v03 = v03;
    tm.v47 = v47;
    return true;
  };
  int max_deg = 1;
  for (int i = 0; i < n; ++i) {
    for (int tt = 0; tt < d->ht_terms; ++tt) {
      const int* rec = d->h_ht_idx + ((size_t)i * d->ht_terms + tt) * d->ht_parts;
      if (!pack(rec, htv, ht[(size_t)tt * n + i])) {
        set_error("hcx_problem_create: dHdt entry (eq %d, term %d) out of range", i, tt);
        return HCX_ERR_INVALID_ARG;
      }
      if (rec[0] != 0) {
        int dg = 0;
        for (int q = 0; q < htv; ++q) dg += rec[2 + q] != n;
        max_deg = std::max(max_deg, dg);
      }
    }
    for (int j = 0; j < n; ++j) {
      for (int tt = 0; tt < d->hx_terms; ++tt) {
        const int* rec = d->h_hx_idx + (((size_t)i * n + j) * d->hx_terms + tt) * d->hx_parts;
        if (!pack(rec, hxv, hx[((size_t)j * d->hx_terms + tt) * n + i])) {
          set_error("hcx_problem_create: dHdx entry (eq %d, var %d, term %d) out of range", i, j, tt);
          return HCX_ERR_INVALID_ARG;
        }
        if (rec[0] != 0) {
          int dg = 1;
          for (int q = 0; q < hxv; ++q) dg += rec[2 + q] != n;
          max_deg = std::max(max_deg, dg);
        }
      }
    }
  }
  // a padded H term still multiplies ht_vars factors; the kernel reads DEG slots
  const int deg = std::max(std::max(max_deg, htv), hxv + 1);
  if (deg > 6) {
    set_error("hcx_problem_create: terms with %d variable factors are not supported (max 6)", deg);
    return HCX_ERR_UNSUPPORTED;
  }

  // LDS slots of the coefficients in the order the lanes of a group read them:
  // dH/dt terms term by term across the equations, then dH/dx terms, then the rest
  std::vector<int> cslot(C + 1, -1), cinv(C + 1, -1);
  int next_slot = 0;
  auto take = [&](dev::Term& tm) {
    if (tm.s == 0) return;
    if (cslot[tm.c] < 0) {
      cslot[tm.c] = next_slot;
      cinv[next_slot] = tm.c;
      ++next_slot;
    }
  };
  for (int tt = 0; tt < d->ht_terms; ++tt)
    for (int i = 0; i < n; ++i) take(ht[(size_t)tt * n + i]);
  for (int j = 0; j < n; ++j)
    for (int tt = 0; tt < d->hx_terms; ++tt)
      for (int i = 0; i < n; ++i) take(hx[((size_t)j * d->hx_terms + tt) * n + i]);
  for (int c = 0; c <= C; ++c)
    if (cslot[c] < 0) {
      cslot[c] = next_slot;
      cinv[next_slot] = c;
      ++next_slot;
    }
  for (auto& tm : ht) tm.c = cslot[tm.c];
  for (auto& tm : hx) tm.c = cslot[tm.c];

  // Term streams (layout and order: hcx_eval.hpp).
  int nslot = 0;  // slots that a term uses come first
  {
    std::vector<char> used(C + 1, 0);
    for (const auto& tm : ht)
      if (tm.s != 0) used[tm.c] = 1;
    for (const auto& tm : hx)
      if (tm.s != 0) used[tm.c] = 1;
    for (int q = 0; q <= C; ++q)
      if (used[q]) nslot = q + 1;
  }
  dev::Term zero_term;
  zero_term.s = 1;
  zero_term.c = 0;
  zero_term.v03 = (uint32_t)(n + 1) | (uint32_t)n << 8 | (uint32_t)n << 16 | (uint32_t)n << 24;
  zero_term.v47 = (uint32_t)n * 0x01010101u;
  // appends one entry's stream [position][equation], up to the last position
  // with a term; returns its scaled positions
  auto add_stream = [&](std::vector<dev::Term>& out, auto&& term_at, int T) {
    int cnt = 0, scaled = 0;
    for (int tt = 0; tt < T; ++tt)
      for (int i = 0; i < n; ++i) {
        const int s = term_at(tt, i).s;
        if (s != 0) cnt = tt + 1;
        if (s != 0 && s != 1) scaled = tt + 1;
      }
    for (int tt = 0; tt < cnt; ++tt)
      for (int i = 0; i < n; ++i) out.push_back(term_at(tt, i).s != 0 ? term_at(tt, i) : zero_term);
    return scaled;
  };
  std::vector<dev::Term> hxs, hts;
  std::vector<int> hxs_cnt(n), ht_ci;
  unsigned int colc[kMaxN] = {};
  bool colc_fits = true;
  int s_min = 0, s_max = 0;
  for (int j = 0; j < n; ++j) {
    const size_t at = hxs.size();
    const int scaled = add_stream(
        hxs, [&](int tt, int i) -> const dev::Term& { return hx[((size_t)j * d->hx_terms + tt) * n + i]; },
        d->hx_terms);
    const size_t cnt = (hxs.size() - at) / n;
    colc_fits = colc_fits && cnt <= 0xffff;
    colc[j] = (unsigned int)(cnt & 0xffff) | ((unsigned int)scaled & 0xffff) << 16;
    hxs_cnt[j] = (int)cnt;
  }
  const int htS = add_stream(
      hts, [&](int tt, int i) -> const dev::Term& { return ht[(size_t)tt * n + i]; }, d->ht_terms);
  const int htT = (int)(hts.size() / n), hx_recs = (int)hxs.size();
  for (const auto& tm : hts) ht_ci.push_back(cinv[tm.c]);
  for (const auto* v : {&hxs, &hts})
    for (const auto& tm : *v) {
      s_min = std::min(s_min, tm.s);
      s_max = std::max(s_max, tm.s);
    }
  if (hxs.empty()) hxs.push_back(zero_term);  // nothing to read, but no empty allocation
  if (hts.empty()) {
    hts.push_back(zero_term);
    ht_ci.push_back(0);
  }
  // compact forms for the instances that hold the streams in LDS
  struct CompactHost {
    std::vector<uint32_t> w;
    int h = 0, slot = 0;
  } compact[6];  // [format], [3 + format]: the latency instances'
  for (int cf = 0; cf < 6; ++cf) {
    const int f = cf % 3;
    const bool lat = cf >= 3;
    // offsets of 16 bits (from the region's start in the slot list), scalars of
    // 6, 16 or 18 bits; the last form where the others do not hold the problem
    const int s_lim = f == 0 ? 32 : (f == 1 ? 32768 : 1 << 17);
    if (!colc_fits || s_min < -s_lim || s_max >= s_lim || nslot > 4000 || C > 0xffff || deg > 2 * f + 2 ||
        (f == 2 && (deg <= 2 || !compact[1].w.empty())))
      continue;
    CompactHost& ch = compact[cf];
    std::vector<uint32_t>& w = ch.w;
    auto var = [&](const dev::Term& tm, int q) {
      return (uint32_t)((((q < 4 ? tm.v03 : tm.v47) >> (8 * (q & 3))) & 0xffu) * 16u);
    };
    auto put = [&](const dev::Term& tm, bool h) {
      const uint32_t sc = (uint32_t)tm.s, j = (uint32_t)cinv[tm.c];
      if (f == 0) {
        w.push_back((uint32_t)(tm.c * 16) | var(tm, 0) << 16 | sc << 26);
        if (h) w.push_back(var(tm, 1) | j << 16);
        return;
      }
      const uint32_t w0 = (uint32_t)(tm.c * 16) | var(tm, 0) << 16, w1 = var(tm, 1) | var(tm, 2) << 16;
      if (f == 2) {
        const uint32_t w2 = var(tm, 3) | var(tm, 4) << 16;
        if (h)
          w.insert(w.end(), {w0 | sc << 26, w1 | sc >> 6 << 26, w2 | sc >> 12 << 26, var(tm, 5) | j << 16});
        else
          w.insert(w.end(), {w0, w1, w2, sc});
        return;
      }
      w.push_back(w0);
      if (h) {
        w.insert(w.end(), {w1, var(tm, 3) | j << 16, sc});
      } else {
        w.push_back(var(tm, 1) | var(tm, 2) << 6 | sc << 16);
      }
    };
    auto align = [&]() {
      while (w.size() % 4) w.push_back(0);
      return (int)(w.size() * 4);
    };
    auto put_lat = [&](const dev::Term& tm) {
      const double sd = tm.s;
      uint64_t bits;
      std::memcpy(&bits, &sd, 8);
      w.push_back((uint32_t)(tm.c * 16) | var(tm, 0) << 16);
      if (f >= 1) w.push_back(var(tm, 1) | var(tm, 2) << 16);
      if (f == 2) w.push_back(var(tm, 3) | var(tm, 4) << 16);
      w.push_back((uint32_t)(bits >> 32));
      if (f == 1) w.push_back(0);
    };
    size_t r = 0;
    for (int j = 0; j < n; ++j) {
      for (int k = 0; k < hxs_cnt[j] * n; ++k, ++r)
        if (lat) put_lat(hxs[r]);
        else put(hxs[r], false);
      for (int i = 0; lat && i < n; ++i) put_lat(zero_term);
    }
    for (int i = 0; !lat && i < n; ++i) put(zero_term, false);  // one row of zero terms for all columns
    ch.h = align();
    r = 0;
    for (int k = 0; k < htT * n; ++k) put(hts[r++], true);
    // a zero term per equation ends the H stream
    for (int i = 0; i < n; ++i) put(zero_term, true);
    ch.slot = align();
    for (int c = 0; c <= C; c += 2) {
      // offsets from the group's region, whose coefficient area follows x and
      // the keys of the instance for n; 0: no slot
      const int head = 16 * (n + 2) + dev::key_bytes(lat || !is_pow2(exact_lanes(n)));
      auto off = [&](int q) { return q > C || cslot[q] >= nslot ? 0u : (uint32_t)(head + cslot[q] * 16); };
      w.push_back(off(c) | off(c + 1) << 16);
    }
    align();
  }

  auto* p = new hcx_problem();
  (void)hipGetDevice(&p->device);
  p->n = n;
  p->C = C;
  p->M = M;
  p->K = d->num_tracks;
  p->k = d->num_params;
  p->hxT = d->hx_terms;
  p->htT_padded = d->ht_terms;
  p->hx_vars = hxv;
  p->ht_vars = htv;
  p->deg = std::max(deg, 2);
  std::memcpy(p->colc, colc, sizeof(colc));
  p->colc_fits = colc_fits;
  p->hx_recs = hx_recs;
  p->htT = htT;
  p->htS = htS;
  p->nslot = nslot;
  p->max_terms = *std::max_element(hxs_cnt.begin(), hxs_cnt.end());
  auto fail = [&](hipError_t e, const char* what) {
    set_error("hcx_problem_create: %s: %s", what, hipGetErrorString(e));
    hcx_problem_destroy(p);
    return HCX_ERR_HIP;
  };
  hipError_t e;
  // every table in one device allocation, filled by one copy
  std::vector<unsigned char> blob;
  std::vector<std::pair<void**, size_t>> parts;
  auto add = [&](auto** dst, const void* src, size_t bytes) {
    parts.emplace_back(reinterpret_cast<void**>(dst), blob.size());
    const unsigned char* c = static_cast<const unsigned char*>(src);
    blob.insert(blob.end(), c, c + bytes);
    blob.resize((blob.size() + 255) & ~size_t(255));
  };
  auto add_vec = [&](auto** dst, const auto& v) { add(dst, v.data(), v.size() * sizeof(v[0])); };
  add_vec(&p->d_cslot, cslot);
  add_vec(&p->d_hx, hxs);
  add_vec(&p->d_ht, hts);
  add_vec(&p->d_ht_ci, ht_ci);
  add_vec(&p->d_hx_cnt, hxs_cnt);
  for (int cf = 0; cf < 6; ++cf) {
    const CompactHost& ch = compact[cf];
    hcx_problem::Compact& ct = cf < 3 ? p->ctab[cf] : p->ltab[cf - 3];
    if (ch.w.empty()) continue;
    add_vec(&ct.d, ch.w);
    ct.words = (int)ch.w.size();
    ct.h = ch.h;
    ct.slot = ch.slot;
  }
  add(&p->d_start, d->h_start_sols, (size_t)p->K * n * sizeof(double2));
  if (p->k > 0 && d->h_coeff_affine) add(&p->d_affine, d->h_coeff_affine, (size_t)C * (1 + p->k) * sizeof(double2));
  if (p->k > 0 && d->h_cmap_scalar) {
    p->cmap_T = d->cmap_terms;
    p->cmap_D = d->cmap_deg;
    const size_t ns = (size_t)C * p->cmap_T;
    add(&p->d_cmap_scalar, d->h_cmap_scalar, ns * sizeof(double2));
    add(&p->d_cmap_params, d->h_cmap_params, ns * p->cmap_D * sizeof(int));
  }
  if (p->k > 0) add(&p->d_p0, d->h_start_params, (size_t)p->k * sizeof(double2));
  // the launcher workspace at the end (nothing to copy)
  const size_t ws_off = blob.size();
  if ((e = hipMalloc(&p->d_blob, ws_off + ws_layout(sizeof(SegOut), 0, 0).bytes)) != hipSuccess)
    return fail(e, "hipMalloc tables");
  if ((e = hipMemcpy(p->d_blob, blob.data(), blob.size(), hipMemcpyHostToDevice)) != hipSuccess)
    return fail(e, "copy tables");
  for (const auto& q : parts) *q.first = p->d_blob + q.second;
  p->launcher_ws.base = p->d_blob + ws_off;

  // algorithmic FLOPs of the reference algorithm (padding terms excluded)
  hcx_problem_info& in = p->info;
  in.num_vars = n;
  in.num_coeffs = C;
  in.max_order_t = M;
  in.num_tracks = p->K;
  in.num_params = p->k;
  in.hx_terms = p->hxT;
  in.ht_terms = p->htT_padded;
  in.hx_vars = hxv;
  in.ht_vars = htv;
  double fh = 0, fhx = 0;
  for (int i = 0; i < n; ++i) {
    for (int tt = 0; tt < d->ht_terms; ++tt) {
      const int* rec = d->h_ht_idx + ((size_t)i * d->ht_terms + tt) * d->ht_parts;
      if (rec[0] == 0) continue;
      int dg = 0;
      for (int q = 0; q < htv; ++q) dg += rec[2 + q] != n;
      fh += f_term(dg);
    }
    for (int j = 0; j < n; ++j)
      for (int tt = 0; tt < d->hx_terms; ++tt) {
        const int* rec = d->h_hx_idx + (((size_t)i * n + j) * d->hx_terms + tt) * d->hx_parts;
        if (rec[0] == 0) continue;
        int dg = 0;
        for (int q = 0; q < hxv; ++q) dg += rec[2 + q] != n;
        fhx += f_term(dg);
      }
  }
  in.flops_coef = (double)C * (8.0 * M - 4.0);
  in.flops_hx = fhx;
  in.flops_ht = fh;
  in.flops_h = fh;
  in.flops_lu = f_lu(n);
  in.flops_stage = in.flops_coef + fhx + fh + in.flops_lu + 16.0 * n;
  in.flops_newton = fhx + fh + in.flops_lu + 12.0 * n;
  *out = p;
  return HCX_OK;
}

hcx_status hcx_problem_destroy(hcx_problem* p) {
  if (!p) return HCX_OK;
  if (p->d_blob) (void)hipFree(p->d_blob);
  delete p;
  return HCX_OK;
}

hcx_status hcx_problem_get_info(const hcx_problem* p, hcx_problem_info* info) {
  clear_error();
  if (!p || !info) {
    set_error("hcx_problem_get_info: null argument");
    return HCX_ERR_INVALID_ARG;
  }
  *info = p->info;
  return HCX_OK;
}

hcx_status hcx_sync(void* stream) {
  clear_error();
  HIP_TRY(hipStreamSynchronize((hipStream_t)stream));
  return HCX_OK;
}

hcx_status hcx_stream_release(void* stream) {
  clear_error();
  if (hcx_device_count() < 1) {
    set_error("hcx_stream_release: no HIP device available");
    return HCX_ERR_NO_DEVICE;
  }
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  return ws_error(pool().release_stream(dev, stream), "hcx_stream_release");
}

// Shared implementation of hcx_track / hcx_track_multi.
}  // extern "C"

namespace hcx {
static thread_local LaunchShape g_shape;

// Shared implementation of hcx_track / hcx_track_multi / graphs / the server.
// `work` (one per segment) is the launch workspace: the stream's pooled
// block, a graph's own block, a server slot's block or the static scratch.
hcx_status track_impl(int nseg, hcx_problem* const* probs, const hcx_batch_desc* batches,
                      const hcx_result_desc* results, const hcx_track_opts* o, hipStream_t stream, int persistent,
                      unsigned long long* batch_start, const LaunchWork* work) {
  hcx_status st = validate_opts(o);
  if (st != HCX_OK) return st;
  if (nseg < 1 || nseg > kMaxSeg || !probs || !batches || !results || !work) {
    set_error("track: need 1..%d segments with problems, batches, results and a workspace", kMaxSeg);
    return HCX_ERR_INVALID_ARG;
  }
  st = ensure_device_info();
  if (st != HCX_OK) return st;
  Launch LN;
  std::memset(&LN, 0, sizeof(LN));
  OutPack OP;
  std::memset(&OP, 0, sizeof(OP));
  LN.nseg = nseg;
  LN.persistent = persistent;
  LN.o = to_opts(o);
  int max_n = 1, max_deg = 2;
  for (int s = 0; s < nseg; ++s) {
    hcx_problem* p = probs[s];
    if (!p) {
      set_error("track: segment %d has no problem", s);
      return HCX_ERR_INVALID_ARG;
    }
    for (int q = 0; q < s; ++q)
      if (probs[q] == p) {
        set_error("track: problem used by two segments of one launch");
        return HCX_ERR_INVALID_ARG;
      }
    max_n = std::max(max_n, p->n);
    max_deg = std::max(max_deg, p->deg);
  }
  int ns[kMaxSeg], Gs[kMaxSeg];
  int specialize = o->specialize;
  bool all_tuned = o->lanes_per_path == 0;
  for (int s = 0; s < nseg; ++s) {
    all_tuned = all_tuned && probs[s]->tuned;
    ns[s] = probs[s]->n;
    if (o->lanes_per_path > 0) Gs[s] = o->lanes_per_path;
    else if (probs[s]->tuned) Gs[s] = probs[s]->tuned_G;
    else Gs[s] = default_lanes(probs[s]->n, probs[s]->C, probs[s]->M);
    if (Gs[s] < ns[s]) {
      set_error("track: lanes_per_path=%d is below n=%d", Gs[s], ns[s]);
      return HCX_ERR_INVALID_ARG;
    }
  }
  if (all_tuned && nseg == 1) specialize = probs[0]->tuned_spec;
  Plan pl;
  st = choose_kernel(nseg, probs, Gs, max_deg, o->precision, specialize, pl);
  if (st != HCX_OK) return st;
  long long total_groups_needed = 0;
  std::vector<long long> seg_groups(nseg);
  for (int s = 0; s < nseg; ++s) {
    hcx_problem* p = probs[s];
    const hcx_batch_desc& b = batches[s];
    const hcx_result_desc& r = results[s];
    // an empty batch (no instances) needs no buffers and tracks nothing
    const bool empty = b.num_instances == 0 || p->K == 0;
    if (b.num_instances < 0 || (!empty && (!r.d_roots || !r.d_flags))) {
      set_error("track: segment %d: bad batch or result descriptor", s);
      return HCX_ERR_INVALID_ARG;
    }
    const int G = Gs[s];
    Seg& S = LN.seg[s];
    SegOut& O = OP.out[s];
    seg_from_problem(S, O, p, G, pl);
    S.I = b.num_instances;
    S.P = (long long)b.num_instances * p->K;
    if (empty) {
      S.chx = nullptr;
      S.cht = nullptr;
    } else if (b.d_coeffs_hx) {
      if (!b.d_coeffs_ht) {
        set_error("track: segment %d: coefficient tables need both Hx and Ht", s);
        return HCX_ERR_INVALID_ARG;
      }
      S.chx = reinterpret_cast<const double2*>(b.d_coeffs_hx);
      S.cht = reinterpret_cast<const double2*>(b.d_coeffs_ht);
    } else {
      if (!b.d_target_params || !b.d_coeff_work || p->k < 1 || (!p->d_cmap_scalar && (!p->d_affine || p->M != 1))) {
        set_error("track: segment %d: needs coefficient tables or target params + a coefficient map + workspace", s);
        return HCX_ERR_INVALID_ARG;
      }
      double2* hx = reinterpret_cast<double2*>(b.d_coeff_work);
      double2* ht = hx + (size_t)b.num_instances * (p->C + 1) * (p->M + 1);
      if (b.num_instances > 0) {
        const double2* p0 = b.d_start_params ? reinterpret_cast<const double2*>(b.d_start_params) : p->d_p0;
        const int p0_stride = b.d_start_params ? p->k : 0;
        dim3 grid((p->C + 1 + 127) / 128, b.num_instances);
        if (p->d_cmap_scalar)
          hipLaunchKernelGGL(p2c_poly_kernel, grid, dim3(128), 0, stream, p->d_cmap_scalar, p->d_cmap_params, p->C,
                             p->cmap_T, p->cmap_D, p->k, p->M, p0, p0_stride,
                             reinterpret_cast<const double2*>(b.d_target_params), b.num_instances, hx, ht);
        else
          hipLaunchKernelGGL(p2c_affine_kernel, grid, dim3(128), 0, stream,
                             reinterpret_cast<const double2*>(p->d_affine), p->C, p->k, p0, p0_stride,
                             reinterpret_cast<const double2*>(b.d_target_params), b.num_instances, hx, ht);
      }
      S.chx = hx;
      S.cht = ht;
    }
    O.roots = reinterpret_cast<double2*>(r.d_roots);
    O.flags = r.d_flags;
    O.steps = r.d_steps;
    O.newton = r.d_newton;
    O.refine = r.d_refine;
    O.tfin = r.d_t_final;
    O.dtfin = r.d_dt_final;
    O.resid = r.d_residual;
    O.inst_done = reinterpret_cast<unsigned long long*>(r.d_inst_done);
    S.counter = work[s].counter;
    S.out = work[s].out;
    O.inst_left = nullptr;
    if (r.d_inst_done && b.num_instances > 0) {
      if (!work[s].inst_left || work[s].inst_cap < b.num_instances) {
        set_error("track: launch workspace instance counters too small (%lld < %d)", work[s].inst_cap,
                  b.num_instances);
        return HCX_ERR_INVALID_ARG;
      }
      O.inst_left = work[s].inst_left;
    }
    if (o->precision == HCX_PREC_MIXED) {
      if (work[s].plist_cap < S.P || !work[s].plist || !work[s].plist_count) {
        set_error("track: launch workspace path list too small (%lld < %lld)", work[s].plist_cap, S.P);
        return HCX_ERR_INVALID_ARG;
      }
      S.plist_count = work[s].plist_count;
    }
    const int gpw = 64 / G;
    seg_groups[s] = (S.P + gpw - 1) / gpw;
    total_groups_needed += seg_groups[s];
  }
  // One-segment FP64 launches of few waves are latency bound: no other waves
  // hide the latency of their evaluations and solves.  They run the latency
  // instance of their size: dc/dt in LDS next to c(t), tables laid out for it,
  // and R replicas of each path's lane group.  In launches of at most one
  // wave per SIMD (or with o->replicas) the replicas split the evaluation's term
  // sums and the solve's columns (the most, a power of two up to 8 with R * G
  // <= 64, that keep the launch within two waves per SIMD, or half of one above
  // R = 2 for light rows), when the group regions and the records fit in 64 KiB.
  // R = 1 takes up to one and a half waves per SIMD (1300 waves: n = 6 2274 -> 2053
  // us, n = 12 4371 -> 4039; at 2048 waves n = 9 loses, 3356 -> 3801).
  bool dealt = false;
  if (o->precision == HCX_PREC_FP64 && nseg == 1) {
    Seg& S = LN.seg[0];
    const hcx_problem* p = probs[0];
    const auto& lat = p->ltab[pl.fmt];
    const int lg = pl.group_bytes(p, true);
    const size_t terms =
        pl.exact ? 0 : ((size_t)p->hx_recs + (size_t)p->n * p->htT) * sizeof(dev::Term);
    Plan lp = pl;
    lp.latency = true;
    auto region = [&](int R) { return ((lp.group_bytes(p, true) + dev::split_bytes(pl.nmax, S.G, R)) / 16 | 1) * 16; };
    auto groups = [&](int R) { return 64 / (S.G * R); };
    auto waves = [&](int R) { return (S.P + groups(R) - 1) / groups(R); };
    const long long w1 = total_groups_needed;
    int R = 1;
    if (o->replicas > 0) {
      R = o->replicas;
      if (R * S.G > 64) {
        set_error("track: %d replicas of %d lanes exceed a wave", R, S.G);
        return HCX_ERR_INVALID_ARG;
      }
    } else if (w1 <= 4LL * g_cu) {
      // at most 8 replicas; beyond 2 and half a wave per SIMD only for rows
      // whose evaluation outweighs the exchange (complex products per row
      // >= 8 per exchanged sum).  The number of replicas is part of the order
      // in which a row's terms are added.
      const int dg = std::max(p->deg, 1);
      const double row_products = (double)p->n * p->hxT * (dg - 1) + (double)p->htT_padded * dg;
      const bool heavy = row_products >= 8.0 * (p->n + 1);
      while (R < 8 && 2 * R * S.G <= 64 && waves(2 * R) <= 8LL * g_cu &&
             (R == 1 || heavy || waves(2 * R) <= 2LL * g_cu))
        R *= 2;
    }
    // the latency instance, also for R = 1
    const bool one = w1 <= 6LL * g_cu;
    const KernelFn rf = one || R > 1 ? pick_rep(pl.nmax, pl.deg, pl.exact, R) : nullptr;
    if (!rf) R = 1;
    const size_t regions = (size_t)groups(R) * (size_t)lg;
    // the rule counts the compact tables of the size-specialised instances at 4
    // or 8 bytes a term, and the full records of the generic ones, which read
    // compact tables where they fit as well
    const bool compact = pl.exact ? pl.tab_lds > 0 : rf && lat.d && lat.words * 4 <= 65536;
    size_t tab = 0, tab_new = terms;
    if (pl.exact && pl.tab_lds > 0) tab = (size_t)table_bytes(p, pl.fmt == 0);
    if (compact) tab_new = (size_t)(rf ? lat.words * 4 : pl.tab_lds);
    const size_t used = (size_t)groups(R) * (size_t)(rf ? region(R) : lg) + tab_new;
    const bool fits = (rf || one) && regions + tab + terms <= 65536 && used <= (size_t)kMaxLdsBytes;
    int deal = 1;
    if ((!fits || R == 1) && o->replicas == 0 && pl.nmax <= 16 && (pl.exact ? pl.tab_lds > 0 : lat.d != nullptr))
      deal = dealt_replicas(S, pl, lat.words * 4, region, waves);
    const KernelFn df = deal > 1 ? pick_deal(pl.nmax, pl.deg, pl.exact, deal) : nullptr;
    if (df && (size_t)groups(deal) * (size_t)region(deal) + (size_t)lat.words * 4 <= (size_t)kMaxLdsBytes) {
      LN.dot_lds = 1;
      dealt = true;
      S.R = deal;
      pl.fn = df;
      pl.latency = true;
      pl.tab_lds = lat.words * 4;
      seg_tables(S, p, pl);
      S.lds_group = region(deal);
      seg_groups[0] = waves(deal);
      total_groups_needed = seg_groups[0];
    } else if (fits) {
      LN.dot_lds = 1;
      S.R = R;
      if (rf) {
        pl.fn = rf;
        pl.latency = true;
        pl.tab_lds = (int)tab_new;
        seg_tables(S, p, pl);
        if (!compact) S.ctab = nullptr;
      }
      S.lds_group = rf ? region(R) : lg;
      seg_groups[0] = waves(R);
      total_groups_needed = seg_groups[0];
    }
  }
  // grid: persistent -> limited by occupancy or the requested waves per CU,
  // split over segments by work
  LN.wpb = 1;
  long long blocks;
  if (persistent) {
    int request = o->waves_per_cu, per_cu = 1;
    if (request == 0 && all_tuned && nseg == 1) request = probs[0]->tuned_wpc;
    const long long waves_needed = std::max<long long>(total_groups_needed, 1);
    st = launch_density(LN, pl, waves_needed, request, per_cu);
    if (st != HCX_OK) return st;
    blocks = std::min<long long>((long long)per_cu * g_cu, (waves_needed + LN.wpb - 1) / LN.wpb);
    // proportional split by estimated work (paths * n^2 as a cost proxy)
    std::vector<double> w(nseg);
    double wsum = 0;
    for (int s = 0; s < nseg; ++s) {
      w[s] = (double)LN.seg[s].P * (double)(probs[s]->n * probs[s]->n + probs[s]->C);
      wsum += w[s];
    }
    long long acc = 0;
    for (int s = 0; s < nseg; ++s) {
      LN.first_block[s] = (int)acc;
      long long nb = wsum > 0 ? (long long)std::llround(blocks * w[s] / wsum) : 0;
      nb = std::min(nb, seg_groups[s]);
      acc += nb;
    }
    LN.first_block[nseg] = (int)acc;
    if (acc < blocks) blocks = std::max<long long>(acc, 1);
    if (acc == 0) blocks = 1;
  } else {
    st = finish_plan(LN, pl);
    if (st != HCX_OK) return st;
    long long acc = 0;
    for (int s = 0; s < nseg; ++s) {
      LN.first_block[s] = (int)acc;
      acc += seg_groups[s];
    }
    LN.first_block[nseg] = (int)acc;
    blocks = std::max<long long>(acc, 1);
  }
  const int wpb = LN.wpb;
  int max_inst = 1;
  for (int s = 0; s < nseg; ++s) max_inst = std::max(max_inst, LN.seg[s].I);
  dim3 ig((max_inst + 255) / 256, nseg);
  hipLaunchKernelGGL(init_kernel, ig, dim3(256), 0, stream, LN, OP, batch_start);
  HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(pl.fn, dim3((unsigned)blocks), dim3(64 * wpb), pl.lds, stream, LN);
  HIP_TRY(hipGetLastError());
  g_shape = {LN.seg[0].R, dealt ? 1 : 0, wpb, (int)blocks, 0, pl.exact ? 1 : 0, pl.tab_lds};

  // Mixed precision: re-track in FP64 from t = 0 every path that ended
  // without a refined root (precision escalation) and every path whose root
  // duplicates another root of its instance (a jump onto another path), then
  // those whose root duplicates a root found by that, so the refined roots and
  // counts are those of the FP64 tracker.
  if (o->precision == HCX_PREC_MIXED) {
    Launch L2 = LN;
    L2.persistent = 1;
    L2.wpb = 1;
    for (int s = 0; s < nseg; ++s) L2.seg[s].plist = work[s].plist;
    Plan p2;
    st = choose_kernel(nseg, probs, Gs, max_deg, HCX_PREC_FP64, specialize, p2);
    if (st != HCX_OK) return st;
    // few paths: latency bound, so dc/dt is staged in LDS when the groups'
    // regions stay within 64 KiB
    size_t need = 0;
    for (int s = 0; s < nseg; ++s)
      need = std::max(need, (size_t)(64 / L2.seg[s].G) * (size_t)p2.group_bytes(probs[s], true));
    if (!p2.exact && need + (size_t)p2.tab_lds > 65536) p2.tab_lds = 0;
    L2.dot_lds = need + (size_t)p2.tab_lds <= 65536 ? 1 : 0;
    for (int s = 0; s < nseg; ++s) {
      seg_tables(L2.seg[s], probs[s], p2);
      L2.seg[s].lds_group = p2.group_bytes(probs[s], L2.dot_lds != 0);
    }
    st = finish_plan(L2, p2);
    if (st != HCX_OK) return st;
    // as many waves as the GPU holds, shared out by the segments' paths: of a
    // batch of diverging paths most are re-tracked (12,288 of n = 12: 40.8 ms on
    // about one wave per CU, 24.1 on all that fit).  The waves that a list
    // has no paths for end at once (run_segment_fp64), so the usual list, of few
    // paths, costs what it did.
    int occ = 0;
    HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, reinterpret_cast<const void*>(p2.fn), 64, p2.lds));
    long long all = 0, b2 = 0;
    for (int s = 0; s < nseg; ++s) all += seg_groups[s];
    const double share = std::min(1.0, (double)std::max(occ, 1) * g_cu / (double)std::max(all, 1LL));
    for (int s = 0; s < nseg; ++s) {
      L2.first_block[s] = (int)b2;
      b2 += std::max<long long>(1, std::llround(share * (double)seg_groups[s]));
    }
    L2.first_block[nseg] = (int)b2;
    g_shape.pass_blocks = (int)b2;
    for (int round = 0; round < (o->retrack_duplicates ? 2 : 1); ++round) {
      for (int s = 0; s < nseg; ++s) L2.seg[s].plist_count = work[s].plist_count + round;
      hipLaunchKernelGGL(list_retrack_kernel, dim3(max_inst, nseg), dim3(256), 0, stream, L2, o->unique_tol, round,
                         o->retrack_duplicates);
      hipLaunchKernelGGL(p2.fn, dim3((unsigned)b2), dim3(64), p2.lds, stream, L2);
    }
    HIP_TRY(hipGetLastError());
  }
  return HCX_OK;
}

}  // namespace hcx

extern "C" {

// The fields of LaunchShape.
void hcx_internal_launch_shape(int* out) { std::memcpy(out, &g_shape, sizeof(g_shape)); }

hcx_status hcx_track(hcx_problem* p, const hcx_batch_desc* b, const hcx_track_opts* o, const hcx_result_desc* r,
                     void* stream) {
  clear_error();
  if (!p || !b || !r) {
    set_error("hcx_track: null argument");
    return HCX_ERR_INVALID_ARG;
  }
  return track_pooled(1, &p, b, r, o, (hipStream_t)stream, 1, reinterpret_cast<unsigned long long*>(r->d_batch_start),
                      "hcx_track");
}

hcx_status hcx_track_multi(int num_segments, hcx_problem* const* problems, const hcx_batch_desc* batches,
                           const hcx_result_desc* results, const hcx_track_opts* o, void* stream) {
  clear_error();
  if (num_segments < 1 || !results) {
    set_error("hcx_track_multi: no segments");
    return HCX_ERR_INVALID_ARG;
  }
  return track_pooled(num_segments, problems, batches, results, o, (hipStream_t)stream, 1,
                      reinterpret_cast<unsigned long long*>(results[0].d_batch_start), "hcx_track_multi");
}

double hcx_kernel_HC_Solver(void* stream, const hcx_problem* pc, int max_steps, int max_corr, int incr_steps,
                            const hcx_complex* d_start_sols, hcx_complex* d_track, const hcx_complex* d_coeffs_hx,
                            const hcx_complex* d_coeffs_ht, uint8_t* d_converge, uint8_t* d_infinity,
                            hcx_complex* d_debug) {
  clear_error();
  hcx_problem* p = const_cast<hcx_problem*>(pc);
  if (!p || !d_start_sols || !d_track || !d_coeffs_hx || !d_coeffs_ht || !d_converge || !d_infinity) {
    set_error("hcx_kernel_HC_Solver: null argument");
    return -1.0;
  }
  hcx_track_opts o;
  hcx_track_opts_default(&o);
  o.max_steps = max_steps;
  o.max_corr = max_corr;
  o.incr_steps = incr_steps;
  o.dt_min = 0.0;
  o.refine_iters = 0;
  if (validate_opts(&o) != HCX_OK) return -1.0;
  if (ensure_device_info() != HCX_OK) return -1.0;
  hipStream_t s = (hipStream_t)stream;
  // the problem's launcher block (counters, output descriptor) serves one
  // synchronous call at a time
  std::lock_guard<std::mutex> lk(p->launcher_mu);
  const LaunchWork w = seg_work(p->launcher_ws, 0, 0, 0);
  Launch LN;
  std::memset(&LN, 0, sizeof(LN));
  OutPack OP;
  std::memset(&OP, 0, sizeof(OP));
  LN.nseg = 1;
  LN.persistent = 0;
  LN.o = to_opts(&o);
  const int G = default_lanes(p->n, p->C, p->M);
  Plan pl;
  if (choose_kernel(1, &p, &G, p->deg, HCX_PREC_FP64, 1, pl) != HCX_OK) return -1.0;
  Seg& S = LN.seg[0];
  SegOut& O = OP.out[0];
  seg_from_problem(S, O, p, G, pl);
  S.start = reinterpret_cast<const double2*>(d_start_sols);
  S.start_stride = p->n + 1;
  O.roots = reinterpret_cast<double2*>(d_track);
  O.roots_stride = p->n + 1;
  S.I = 1;
  S.P = p->K;
  S.chx = reinterpret_cast<const double2*>(d_coeffs_hx);
  S.cht = reinterpret_cast<const double2*>(d_coeffs_ht);
  S.counter = w.counter;
  S.out = w.out;
  // the reference's outputs only: converged / infinity bytes and (t, dt)
  O.flags = nullptr;
  O.conv8 = d_converge;
  O.inf8 = d_infinity;
  O.debug = reinterpret_cast<double2*>(d_debug);
  const int gpw = 64 / G;
  LN.first_block[0] = 0;
  LN.first_block[1] = (p->K + gpw - 1) / gpw;
  if (finish_plan(LN, pl) != HCX_OK) return -1.0;
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
    set_error("hcx_kernel_HC_Solver: hipEventCreate failed");
    return -1.0;
  }
  hipLaunchKernelGGL(init_kernel, dim3(1, 1), dim3(64), 0, s, LN, OP, (unsigned long long*)nullptr);
  (void)hipEventRecord(e0, s);
  hipLaunchKernelGGL(pl.fn, dim3(LN.first_block[1]), dim3(64), pl.lds, s, LN);
  hipError_t le = hipGetLastError();
  (void)hipEventRecord(e1, s);
  hipError_t se = hipEventSynchronize(e1);
  float ms = 0.f;
  (void)hipEventElapsedTime(&ms, e0, e1);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (le != hipSuccess || se != hipSuccess) {
    set_error("hcx_kernel_HC_Solver: launch failed: %s", hipGetErrorString(le != hipSuccess ? le : se));
    return -1.0;
  }
  return ms * 1e-3;
}

// hcx_track with the static scratch as its launch workspace: nothing is
// allocated (no hipMalloc, no pool, no allocating library call).
hcx_status hcx_track_noalloc(hcx_problem* p, const hcx_batch_desc* b, const hcx_track_opts* o,
                             const hcx_result_desc* r, void* stream) {
  clear_error();
  if (!p || !b || !r || !o) {
    set_error("hcx_track_noalloc: null argument");
    return HCX_ERR_INVALID_ARG;
  }
  long long inst = 0, paths = 0;
  ws_need(1, &p, b, r, o, inst, paths);
  if (inst > HCX_NOALLOC_MAX_INSTANCES || paths > HCX_NOALLOC_MAX_PATHS) {
    set_error("hcx_track_noalloc: the batch needs %lld instance counters and %lld re-track entries; the static "
              "scratch holds %d and %d", inst, paths, HCX_NOALLOC_MAX_INSTANCES, HCX_NOALLOC_MAX_PATHS);
    return HCX_ERR_INVALID_ARG;
  }
  WsBlock blk;
  hcx_status st = scratch_block(blk);
  if (st != HCX_OK) return st;
  LaunchWork work[1];
  ws_carve(blk, 1, b, r, &p, o, work);
  return track_impl(1, &p, b, r, o, (hipStream_t)stream, 1, reinterpret_cast<unsigned long long*>(r->d_batch_start),
                    work);
}

// Reference-style per-instance launch with the generic result layout (no
// persistence, no refill): used as the plain per-problem baseline.
hcx_status hcx_track_static(hcx_problem* p, const hcx_batch_desc* b, const hcx_track_opts* o,
                            const hcx_result_desc* r, void* stream) {
  clear_error();
  if (!p || !b || !r) {
    set_error("hcx_track_static: null argument");
    return HCX_ERR_INVALID_ARG;
  }
  return track_pooled(1, &p, b, r, o, (hipStream_t)stream, 0, reinterpret_cast<unsigned long long*>(r->d_batch_start),
                      "hcx_track_static");
}

hcx_status hcx_collect(int n, int num_instances, int num_tracks, const hcx_complex* d_roots, uint32_t* d_flags,
                       double unique_tol, hcx_counts* out, void* stream) {
  clear_error();
  const bool empty = num_instances == 0 || num_tracks == 0;
  if (n < 1 || num_instances < 0 || num_tracks < 0 || (!empty && (!d_roots || !d_flags)) || !out) {
    set_error("hcx_collect: invalid arguments");
    return HCX_ERR_INVALID_ARG;
  }
  // bit sets, then the instance's roots when they fit in 48 KiB of LDS
  const size_t bit_lds = 16 * (size_t)((4 * ((num_tracks + 31) / 32) + 3) / 4);
  const size_t root_lds = sizeof(double2) * (size_t)num_tracks * n;
  if (bit_lds > 65536) {
    set_error("hcx_collect: %d paths per instance exceed the collection kernel's bit sets", num_tracks);
    return HCX_ERR_UNSUPPORTED;
  }
  const int stage = bit_lds + root_lds <= 48 * 1024 ? 1 : 0;
  const size_t lds = bit_lds + (stage ? root_lds : 0);
  hcx_status st = ensure_device_info();
  if (st != HCX_OK) return st;
  std::lock_guard<std::mutex> lk(g_mu);
  if (!g_counts) HIP_TRY(hipMalloc(&g_counts, kNumCounts * sizeof(unsigned long long)));
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(zero_u64_kernel, dim3(1), dim3(64), 0, s, g_counts, kNumCounts);
  if (!empty)
    hipLaunchKernelGGL(collect_kernel, dim3(num_instances), dim3(256), lds, s, n, num_tracks,
                       reinterpret_cast<const double2*>(d_roots), d_flags, unique_tol, g_counts, stage);
  HIP_TRY(hipGetLastError());
  unsigned long long h[kNumCounts];
  HIP_TRY(hipMemcpyAsync(h, g_counts, sizeof(h), hipMemcpyDeviceToHost, s));
  HIP_TRY(hipStreamSynchronize(s));
  out->tracked = (int64_t)h[0];
  out->infinity = (int64_t)h[1];
  out->refined = (int64_t)h[2];
  out->real = (int64_t)h[3];
  out->unique = (int64_t)h[4];
  out->unique_ref = (int64_t)h[5];
  out->real_ref = (int64_t)h[6];
  return HCX_OK;
}

}  // extern "C"

// ============================================================== autotuner + graphs
extern "C" {

// Times candidate launch shapes of problem p on a sample batch and keeps the
// fastest: lanes per path G in {n, next power of two <= 64}, the
// size-specialised or the generic kernel instance, and the persistent grid
// density (occupancy, half occupancy).  Results are bitwise-independent of
// the grid density; G and the kernel variant change only the summation order
// of group reductions.
hcx_status hcx_autotune(hcx_problem* p, const hcx_batch_desc* sample, const hcx_track_opts* o,
                        hcx_tune_result* out, void* stream) {
  clear_error();
  if (!p || !sample || !o || sample->num_instances < 1) {
    set_error("hcx_autotune: need a problem, options and a non-empty sample batch");
    return HCX_ERR_INVALID_ARG;
  }
  hcx_status st = validate_opts(o);
  if (st != HCX_OK) return st;
  hipStream_t s = (hipStream_t)stream;
  const long long P = (long long)sample->num_instances * p->K;
  double2* roots = nullptr;
  uint32_t* flags = nullptr;
  HIP_TRY(hipMalloc(&roots, sizeof(double2) * P * p->n));
  HIP_TRY(hipMalloc(&flags, sizeof(uint32_t) * P));
  hcx_result_desc r;
  std::memset(&r, 0, sizeof(r));
  r.d_roots = reinterpret_cast<hcx_complex*>(roots);
  r.d_flags = flags;
  const int G0 = default_lanes(p->n, p->C, p->M);
  int pow2 = 1;
  while (pow2 < G0) pow2 <<= 1;
  struct Cand { int G, spec, wpc; };
  std::vector<Cand> cands;
  int occ = 0;
  {
    // waves per CU of the default shape, to derive the half-density candidate
    Plan pl;
    int G = G0;
    if (choose_kernel(1, &p, &G, p->deg, o->precision, 1, pl) == HCX_OK) {
      Launch LN;
      std::memset(&LN, 0, sizeof(LN));
      SegOut O;
      LN.nseg = 1;
      seg_from_problem(LN.seg[0], O, p, G, pl);
      int nb = 0;
      if (ensure_device_info() == HCX_OK &&
          launch_density(LN, pl, (P + 64 / G - 1) / (64 / G), 0, nb) == HCX_OK)
        occ = nb * LN.wpb;
    }
  }
  for (int spec = 1; spec >= (G0 == p->n ? 0 : 1); --spec) {
    cands.push_back({G0, spec, 0});
    if (occ > 1) cands.push_back({G0, spec, std::max(1, occ / 2)});
  }
  if (pow2 != G0 && pow2 <= 64) {
    cands.push_back({pow2, 0, 0});
    if (occ > 1) cands.push_back({pow2, 0, std::max(1, occ / 2)});
  }
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0));
  HIP_TRY(hipEventCreate(&e1));
  double best = 1e300;
  Cand bc = cands[0];
  const bool was_tuned = p->tuned;
  p->tuned = false;
  int timed = 0;
  for (const Cand& c : cands) {
    hcx_track_opts oc = *o;
    oc.lanes_per_path = c.G;
    oc.specialize = c.spec;
    oc.waves_per_cu = c.wpc;
    st = track_pooled(1, &p, sample, &r, &oc, s, 1, nullptr, "hcx_autotune");  // warm-up
    if (st != HCX_OK) continue;
    HIP_TRY(hipEventRecord(e0, s));
    const int reps = 2;
    for (int q = 0; q < reps && st == HCX_OK; ++q)
      st = track_pooled(1, &p, sample, &r, &oc, s, 1, nullptr, "hcx_autotune");
    HIP_TRY(hipEventRecord(e1, s));
    HIP_TRY(hipEventSynchronize(e1));
    if (st != HCX_OK) continue;
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
    ++timed;
    if (ms / reps < best) {
      best = ms / reps;
      bc = c;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  (void)hipFree(roots);
  (void)hipFree(flags);
  if (timed == 0) {
    p->tuned = was_tuned;
    char msg[512];
    std::snprintf(msg, sizeof(msg), "%s", hcx_last_error());
    set_error("hcx_autotune: no candidate ran (%s)", msg);
    return HCX_ERR_UNSUPPORTED;
  }
  p->tuned = true;
  p->tuned_G = bc.G;
  p->tuned_spec = bc.spec;
  p->tuned_wpc = bc.wpc;
  if (out) {
    out->lanes_per_path = bc.G;
    out->specialize = bc.spec;
    out->waves_per_cu = bc.wpc;
    out->best_ms = best;
    out->candidates = timed;
  }
  return HCX_OK;
}

hcx_status hcx_problem_set_launch_shape(hcx_problem* p, int lanes_per_path, int specialize, int waves_per_cu) {
  clear_error();
  if (!p || lanes_per_path < 0 || lanes_per_path > 64 || (lanes_per_path > 0 && lanes_per_path < p->n) ||
      specialize < 0 || specialize > 1 || waves_per_cu < 0) {
    set_error("hcx_problem_set_launch_shape: invalid shape");
    return HCX_ERR_INVALID_ARG;
  }
  p->tuned = lanes_per_path > 0;
  p->tuned_G = lanes_per_path;
  p->tuned_spec = specialize;
  p->tuned_wpc = waves_per_cu;
  return HCX_OK;
}

}  // extern "C"

struct hcx_graph {
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  // the graph's own launch workspace (path queues, output descriptors,
  // instance counters, re-track list): baked into the graph, freed with it
  WsBlock ws;
  hipEvent_t last = nullptr;  // completion of the latest replay
};

extern "C" {

// Captures one multi-segment persistent launch (counter set-up, device P2C,
// tracking, and in mixed precision the FP64 re-track pass) into a HIP graph.
// Counters are cleared by kernels, not memset nodes.  The arguments are baked
// into the graph: the same device buffers are reused on every
// hcx_graph_launch.  The launch workspace belongs to the graph, so eager
// launches of the same problems on any stream, of any size, never touch the
// memory a replay uses.
hcx_status hcx_graph_capture_multi(int num_segments, hcx_problem* const* problems, const hcx_batch_desc* batches,
                                   const hcx_result_desc* results, const hcx_track_opts* o, hcx_graph** out) {
  clear_error();
  if (!out || num_segments < 1 || num_segments > kMaxSeg || !problems || !batches || !results || !o) {
    set_error("hcx_graph_capture_multi: invalid arguments");
    return HCX_ERR_INVALID_ARG;
  }
  for (int s = 0; s < num_segments; ++s)
    if (!problems[s]) {
      set_error("hcx_graph_capture_multi: segment %d has no problem", s);
      return HCX_ERR_INVALID_ARG;
    }
  auto* g = new hcx_graph();
  long long inst = 0, paths = 0;
  ws_need(num_segments, problems, batches, results, o, inst, paths);
  const WsLayout L = ws_layout(sizeof(SegOut), inst, paths);
  hipError_t e = hipMalloc(&g->ws.base, L.bytes);
  if (e != hipSuccess) {
    delete g;
    set_error("hcx_graph_capture_multi: workspace allocation: %s", hipGetErrorString(e));
    return HCX_ERR_OUT_OF_MEMORY;
  }
  g->ws.inst_cap = inst;
  g->ws.paths_cap = paths;
  g->ws.pinned = true;
  LaunchWork work[kMaxSeg];
  ws_carve(g->ws, num_segments, batches, results, problems, o, work);
  // an uncaptured run first: sets kernel attributes outside the capture
  hipStream_t cs = nullptr;
  hcx_status st = HCX_OK;
  if ((e = hipStreamCreateWithFlags(&cs, hipStreamNonBlocking)) != hipSuccess ||
      (e = hipEventCreateWithFlags(&g->last, hipEventDisableTiming)) != hipSuccess) {
    set_error("hcx_graph_capture_multi: %s", hipGetErrorString(e));
    st = HCX_ERR_HIP;
  }
  if (st == HCX_OK)
    st = track_impl(num_segments, problems, batches, results, o, cs, 1,
                    reinterpret_cast<unsigned long long*>(results[0].d_batch_start), work);
  if (st == HCX_OK && (e = hipStreamSynchronize(cs)) != hipSuccess) {
    set_error("hcx_graph_capture_multi: %s", hipGetErrorString(e));
    st = HCX_ERR_HIP;
  }
  if (st == HCX_OK) {
    e = hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal);
    if (e == hipSuccess) {
      st = track_impl(num_segments, problems, batches, results, o, cs, 1,
                      reinterpret_cast<unsigned long long*>(results[0].d_batch_start), work);
      hipError_t e2 = hipStreamEndCapture(cs, &g->graph);
      if (st == HCX_OK && e2 != hipSuccess) {
        set_error("hipStreamEndCapture: %s", hipGetErrorString(e2));
        st = HCX_ERR_HIP;
      }
    } else {
      set_error("hipStreamBeginCapture: %s", hipGetErrorString(e));
      st = HCX_ERR_HIP;
    }
  }
  if (st == HCX_OK) {
    e = hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0);
    if (e != hipSuccess) {
      set_error("hipGraphInstantiate: %s", hipGetErrorString(e));
      st = HCX_ERR_HIP;
    }
  }
  if (cs) (void)hipStreamDestroy(cs);
  if (st != HCX_OK) {
    hcx_graph_destroy(g);
    return st;
  }
  *out = g;
  return HCX_OK;
}

hcx_status hcx_graph_launch(hcx_graph* g, void* stream) {
  clear_error();
  if (!g || !g->exec) {
    set_error("hcx_graph_launch: no graph");
    return HCX_ERR_INVALID_ARG;
  }
  HIP_TRY(hipGraphLaunch(g->exec, (hipStream_t)stream));
  HIP_TRY(hipEventRecord(g->last, (hipStream_t)stream));
  return HCX_OK;
}

// Waits for the latest replay, then frees the graph and its workspace.
hcx_status hcx_graph_destroy(hcx_graph* g) {
  if (!g) return HCX_OK;
  if (g->last) {
    (void)hipEventSynchronize(g->last);
    (void)hipEventDestroy(g->last);
  }
  if (g->exec) (void)hipGraphExecDestroy(g->exec);
  if (g->graph) (void)hipGraphDestroy(g->graph);
  if (g->ws.base) (void)hipFree(g->ws.base);
  delete g;
  return HCX_OK;
}

}  // extern "C"
