// Tracker kernel templates (shared by the per-instance translation units).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "hcx_device.hpp"
#include "hcx_flags.h"

namespace hcx {

using dev::cx;
using dev::cmk;

constexpr int kMaxSeg = 8;
constexpr int kMaxN = 32;
// terms whose table records are requested together when the tables are read
// from global memory
#ifndef HCX_TERM_CHUNK
#define HCX_TERM_CHUNK 4
#endif
constexpr int kTermChunk = HCX_TERM_CHUNK;
// Lanes per path of the size-specialised instance for n: n, except n = 30,
// which runs on aligned 32-lane groups (still two paths per wave) so that
// its group reductions can use DPP row permutations.
constexpr int exact_lanes(int n) { return n == 30 ? 32 : n; }
constexpr bool is_pow2(int g) { return g > 0 && (g & (g - 1)) == 0; }

// Output pointers of a segment (cold): kept in device memory and read only
// when a path finishes, so they do not occupy scalar registers in the loop.
struct SegOut {
  double2* roots;              // [P][roots_stride]
  uint32_t* flags;
  int* steps;
  int* newton;
  int* refine;
  double* tfin;
  double* dtfin;
  double* resid;
  uint8_t* conv8;
  uint8_t* inf8;
  double2* debug;
  unsigned long long* inst_done;
  int* inst_left;
  int roots_stride;
};

// Per-launch device workspace of one segment (path queue, output
// descriptor, per-instance remaining-path counters, re-track path list).
struct LaunchWork {
  unsigned int* counter;
  SegOut* out;
  int* inst_left;              // capacity inst_cap
  int* plist;                  // re-track path list (capacity plist_cap)
  unsigned int* plist_count;   // [2], one per round of the re-track pass
  long long inst_cap;
  long long plist_cap;
};

// Hot, wave-uniform description of one segment (kernel arguments).
struct Seg {
  int n, C, M, K;
  int htT;
  int G;
  int R;                       // replicas per path (lanes per path = G * R; FP64 loop)
  int lds_group;               // bytes of one group's LDS region
  int start_stride;
  int I;
  long long P;
  const dev::Term* hx;         // term streams (hcx_eval.hpp), full records
  const dev::Term* ht;
  // per Jacobian column: positions of its stream | scaled ones << 16; where a
  // number does not fit, hx_cnt (device memory) holds the positions instead
  // (else nullptr)
  unsigned int colc[kMaxN];
  const int* hx_cnt;
  const int* ht_ci;            // coefficient numbers of the ht records
  // scaled positions of ht (htT: all); records of hx; coefficients with an
  // LDS slot
  int htS, hx_recs, nslot;
  int max_terms;               // positions of the longest column
  int tab_words;               // 4-byte words of the compact tables
  int tab_h, tab_slot;         // byte offsets of their H streams and slot list
  const double2* start;        // [K][start_stride]
  const double2* chx;          // [I][C+1][M+1]
  const double2* cht;          // [I][C+1][M]
  const int* cslot;            // [C+1] LDS slot of coefficient j (the tables hold slots)
  const uint32_t* ctab;        // compact tables (instances that hold the streams in LDS)
  unsigned int* counter;
  const SegOut* out;           // device copy written by init_kernel
  int* plist;                  // optional: track only these paths (count in *plist_count)
  unsigned int* plist_count;   // mixed: set in the first launch too, whose set-up clears the counts
};

struct Opts {
  int max_steps, max_corr, incr, refine_iters;
  int newton32;      // mixed: FP32 corrector before the end zone
  double dt0, t_tol, dt_min, corr_tol, inf_tol, refine_tol, real_tol;
  double real_ref_tol;  // the reference's real test on the tracked root
  double ez_enter;   // enter the end zone when |1 - t| <= end_zone + 1e-7
  double ez_land;    // before the end zone, steps land on 1 - end_zone
};

struct Launch {
  Seg seg[kMaxSeg];
  int nseg;
  int first_block[kMaxSeg + 1];
  int persistent;
  int tab_lds;                 // bytes of dynamic LDS before the group regions (compact tables)
  int dot_lds;                 // FP64 mode, M = 1: stage dc/dt in LDS (else read it from global)
  int wpb;                     // waves per block (> 1 only for one-segment launches: the
                               // waves of a block share one copy of the compact tables)
  Opts o;
};

// The options and segment descriptors in the kernel-argument (constant)
// address space: loads through these types are scalar loads.
typedef const __attribute__((address_space(4))) Opts KOpts;
typedef const __attribute__((address_space(4))) Seg KSeg;

}  // namespace hcx

#include "hcx_eval.hpp"

namespace hcx {
namespace dev {

// The launch's options where the kernel argument holds them (the
// descriptor is the kernels' only argument: offset 0 of the segment).
__device__ __forceinline__ const KOpts* launch_opts() {
  return (const KOpts*)((const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr() +
                        offsetof(Launch, o));
}

// Segment si's descriptor where the kernel argument holds it.
__device__ __forceinline__ const KSeg* launch_seg(int si) {
  return (const KSeg*)((const __attribute__((address_space(4))) char*)__builtin_amdgcn_kernarg_segment_ptr() +
                       offsetof(Launch, seg) + (size_t)si * sizeof(Seg));
}

// A kernel-argument view for one iteration of a path loop: the pointer
// passes through an empty asm keyed on the iteration count, so the fields
// are re-read (scalar loads) where an iteration uses them instead of
// staying live in scalar registers across the loop, where they would be
// spilled to vector-register lanes and reloaded with VALU instructions.
template <class T>
__device__ __forceinline__ T* iteration_view(T* p, int iter) {
  asm("" : "+s"(p) : "s"(iter));
  return p;
}

template <class T>
__device__ __forceinline__ T group_max(T v, const Group& g) {
  for (int s = 1; s < g.G; s <<= 1) {
    int src = g.gl + s;
    src = (src >= g.G ? src - g.G : src) + g.gbase;
    const T o = lane_read(v, src);
    v = o > v ? o : v;
  }
  return v;
}

// Pivot key of a candidate row: its magnitude's bits above 31 - label, so the
// largest key is the largest magnitude and, among equal ones, the first row in
// current row order.  A row that is no candidate holds key 0; NaN orders above
// every number.  An FP32 key is two words and holds the whole magnitude (0: a key below 32).
// An FP64 key is one word, the upper 27 bits without the sign.  Where candidates
// share these (one pair in 2^16 of unrelated ones, and exact ties), the key's
// pivot is compared with them, and a larger one is found in a second search over
// the other bits and the label (pivot_rest), so the pivot is that of the whole
// magnitudes.
__device__ __forceinline__ unsigned long long pivot_key(float mag, int label) {
  return ((unsigned long long)(__float_as_uint(mag) & 0x7fffffffu) << 32) | (unsigned int)(31 - label);
}
__device__ __forceinline__ unsigned int pivot_key(double mag, int label) {
  return ((unsigned int)((unsigned long long)__double_as_longlong(mag) >> 31) & ~31u) | (unsigned int)(31 - label);
}
// The bits that the FP64 key leaves out, above 31 - label; bit 63 is set.
__device__ __forceinline__ unsigned long long pivot_rest(double mag, int label) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(mag) & ((1ull << 36) - 1);
  return 1ull << 63 | b << 5 | (unsigned int)(31 - label);
}
// A group's key words hold one kind or the other.
typedef unsigned int __attribute__((may_alias)) key32;
typedef unsigned long long __attribute__((may_alias)) key64;
// A group has few of them, used in turn and cleared together when the steps
// come round (every step's result has been read by then): a word per step took
// up to 256 bytes of a region, which refused problems of the widest tables.
constexpr int kKeyWords = 4;
__device__ __forceinline__ void clear_keys(unsigned long long* keys, const Group& g, bool row) {
  if (row && g.s == 0 && g.gl < kKeyWords) keys[g.gl] = 0ull;
  HCX_WAVE_SYNC();
}
__device__ __forceinline__ bool same_upper(unsigned int a, unsigned int b) { return (a ^ b) < 32u; }
// Whether a search of the wave is still open: more than one candidate shares a
// key's upper bits, or these are 0 (the group's other lanes hold key 0).  One
// scalar branch.  part: the lanes of the paths that take part, searches: their
// number (-1 where a path has one lane).
__device__ __forceinline__ bool pivot_open(unsigned int own, unsigned int key, unsigned long long part, int searches) {
  return (int)__builtin_popcountll(__ballot(same_upper(own, key)) & part) != searches;
}

// Largest value over an aligned group of GC lanes (a power of two), to every
// lane: DPP inside 16-lane rows, a row swap between the two rows of 32.
template <int CTRL>
__device__ __forceinline__ unsigned int max_dpp(unsigned int k) {
  return max(k, (unsigned int)dpp_read<CTRL>((int)k));
}
template <int CTRL>
__device__ __forceinline__ unsigned long long max_dpp(unsigned long long k) {
  const unsigned int lo = (unsigned int)dpp_read<CTRL>((int)(unsigned int)k);
  const unsigned int hi = (unsigned int)dpp_read<CTRL>((int)(unsigned int)(k >> 32));
  return max(k, ((unsigned long long)hi << 32) | lo);
}
// rows (0, 0, 2, 2) and (1, 1, 3, 3) of the wave
__device__ __forceinline__ unsigned int max_rows(unsigned int k) {
  const auto r = __builtin_amdgcn_permlane16_swap(k, k, false, false);
  return max((unsigned int)r[0], (unsigned int)r[1]);
}
__device__ __forceinline__ unsigned long long max_rows(unsigned long long k) {
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned int)k, (unsigned int)k, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned int)(k >> 32), (unsigned int)(k >> 32), false, false);
  return max(((unsigned long long)hi[0] << 32) | lo[0], ((unsigned long long)hi[1] << 32) | lo[1]);
}
template <int GC, class K>
__device__ __forceinline__ K group_max_key(K k) {
  static_assert(is_pow2(GC) && GC <= 32, "aligned power-of-two groups");
  if constexpr (GC >= 2) k = max_dpp<kDppQuadXor1>(k);
  if constexpr (GC >= 4) k = max_dpp<kDppQuadXor2>(k);
  if constexpr (GC >= 8) k = max_dpp<kDppHalfMirror>(k);
  if constexpr (GC >= 16) k = max_dpp<kDppRowMirror>(k);
  if constexpr (GC >= 32) k = max_rows(k);
  return k;
}

// Sums over the group's rows of two per-row values (the corrector's and the
// refinement's |d|^2 and |x|^2), returned to every lane of the group.  Aligned
// power-of-two groups use lane exchanges; other group sizes publish the
// pairs in the group's LDS slots `q` and every lane adds them, in row order
// (TREE: in pairs, pairs of pairs, ..., the order of the lane exchanges), for
// one LDS round trip where the exchanges are ten.
template <int NMAX, int GC, bool TREE>
__device__ __forceinline__ void group_sum2(double& a, double& b, const Group& g, int n, bool row, int lane,
                                           cx<double>* q) {
  if constexpr (GC > 0 || (TREE && NMAX > 16)) {
    a = group_sum(a, g, lane);
    b = group_sum(b, g, lane);
  } else {
    if (row) q[g.gl] = cmk<double>(a, b);
    HCX_WAVE_SYNC();
    if constexpr (TREE) {
      cx<double> v[NMAX];
#pragma unroll
      for (int j = 0; j < NMAX; ++j) v[j] = j < n ? q[j] : cmk<double>(0, 0);
#pragma unroll
      for (int w = 1; w < NMAX; w <<= 1)
#pragma unroll
        for (int j = 0; j + w < NMAX; j += 2 * w) v[j] = cadd(v[j], v[j + w]);
      HCX_WAVE_SYNC();
      a = v[0].re;
      b = v[0].im;
    } else {
      double sa = 0.0, sb = 0.0;
#pragma unroll
      for (int j = 0; j < NMAX; ++j) {
        if (j < n) {
          const cx<double> v = q[j];
          sa += v.re;
          sb += v.im;
        }
      }
      HCX_WAVE_SYNC();
      a = sa;
      b = sb;
    }
  }
}

// ------------------------------------------------------------ group solve
// Solves A x = b for the group's n x n system, row r held by lane r (A[j] =
// A[r][j]).  Returns x_gl to lane gl.  Pivoting is the reference's partial
// pivoting (dev-cgesv-batched-small.cuh:51-95): cabs1, the first maximum in
// current row order (rows carry a position label swapped like a physical
// row interchange), multipliers by the pivot reciprocal, a zero pivot column
// reported through `singular`.  Every step eliminates the pivot
// column from the rows ABOVE the pivot as well (Gauss-Jordan), in place of the
// reference's back substitution (:97-106): on a lane group the lanes of those
// rows would only wait during the step, so the extra row updates cost no
// issue cycles, while the n-step dependent chain of the back substitution
// (a lane exchange per step) and the need to keep U alive for it disappear
// (n = 30 FP64: 157 instead of about 290 registers).  The candidate rows of
// each pivot search receive exactly the updates of the LU, so the pivot
// sequence is the LU's.  At the end the lane holding position i has
// x_i = b_i / U_ii; one LDS exchange returns x_gl to lane gl.  A zero pivot
// makes every component NaN (the reference's division by a zero U_ii gives
// NaN in that component and in the rows that depend on it; the tracker only
// reacts to whether any component is not finite).
//
// The solve is a chain of n steps, each bound by its latencies: find the
// pivot, broadcast its row, update.  So
//  * a candidate packs its magnitude and position into one key; the largest
//    comes from DPP row permutations (aligned power-of-two groups) or from an
//    LDS maximum per group and step (one instruction and one read in place of
//    a scan of every candidate's magnitude);
//  * whether an FP64 key left candidates to compare further (pivot_open) is
//    looked at while the pivot's row is on its way; if a larger one is found the
//    row goes out again.  Against keys of 59 bits that called the rest equal:
//    lone launches of n = 3 and 5 +0.2 and +1.1%, n = 12 -0.8%, n = 30 -3.1%
//    (DPP steps on one word); generalized_3views_4pts, whose columns hold equal
//    magnitudes at most steps, 1.31 -> 1.39 ms (1.47 with a second search for
//    every tie);
//  * the next step's candidates enter their search as soon as their column is
//    updated, and the remaining columns are updated while it is under way;
//  * every candidate computes the reciprocal of its own entry during the
//    search, and the pivot's goes out with its row.
// keys: kKeyWords LDS words of the group (unused with GC > 0).
// Where n is not a compile-time constant (generic instances) the columns are
// checked against it four at a time: columns n..NMAX-1 hold values that no
// step uses.
// act: the group's path takes part (the others' results are not used).
template <int NMAX, int GC, class T>
__device__ __forceinline__ cx<T> group_lu_solve(cx<T> (&A)[NMAX], cx<T> b, const Group& g, int n, bool row, bool act,
                                                cx<T>* sp, unsigned long long* keys, bool& singular) {
  const unsigned long long part = __ballot(act);
  const int searches = g.G == 1 ? -1 : __popcll(__ballot(act && g.gl == 0));  // one per path and replica
  int label = g.gl;
  cx<T> own_rinv = cmk<T>(T(0), T(0));  // 1 / U_ii of the row this lane ends up holding
  singular = false;
  // Every lane takes part in the LDS maximum (a mask would cost a branch): a
  // lane that is no candidate, or belongs to a replica other than the first
  // (whose rows are replica 0's), adds key 0, which changes no word, to a word
  // of its own among the group's x slots.
  constexpr int kXWords = 2 * (NMAX + 2);
  unsigned long long* const no_key = keys - kXWords + (g.gl + g.s * g.G) % kXWords;
  if constexpr (GC == 0) clear_keys(keys, g, row);
  // sp shares the group's LDS slots with x: the evaluation's reads of x come first
  HCX_WAVE_SYNC();
  // the group's largest key for step k, and this lane's
  decltype(pivot_key(T(0), 0)) key = 0, own = 0;
  auto largest = [&](int k, bool in, auto v) {
    using V = decltype(v);
    using W = std::conditional_t<sizeof(V) == 4, key32, key64>;
    if constexpr (GC > 0) return group_max_key<GC>(in ? v : V(0));
    const bool mine = in && g.s == 0;
    __hip_atomic_fetch_max(reinterpret_cast<W*>(mine ? &keys[k % kKeyWords] : no_key), mine ? v : V(0), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WAVEFRONT);
    // requested ahead of the rest of the pivot row
    HCX_WAVE_SYNC();
    const V m = *reinterpret_cast<W*>(&keys[k % kKeyWords]);
    HCX_WAVE_SYNC();
    return m;
  };
  auto search = [&](int k) {
    const bool cand = row && label >= k;
    own = cand ? pivot_key(cabs1(A[k]), label) : 0;
    key = largest(k, cand, own);
  };
  search(0);
#pragma unroll
  for (int k = 0; k < NMAX; ++k) {
    if (k < n) {
      cx<T> rinv = crecip(A[k]);
      // keeps the reciprocal out of the pivot's branch, beside the search
      asm volatile("" : "+v"(rinv.re), "+v"(rinv.im));
      int blabel = 31 - (int)((unsigned int)key & 31u);
      if constexpr (sizeof(T) == 4) singular = singular || key < 32;
      bool piv = row && label == blabel;
      const bool more = k + 1 < NMAX && k + 1 < n;
      // the two entries that the next search waits for go out, and are
      // requested, before the rest of the row
      constexpr bool kSplit = NMAX > 6;
      cx<T> rp, next = cmk<T>(T(0), T(0));
      auto publish = [&]() {
        if (piv) {
          sp[k] = rinv;
          if (more) sp[k + 1] = A[k + 1];
          if constexpr (!kSplit) {
#pragma unroll
            for (int j = k + 2; j < NMAX; ++j)
              if ((j & ~3) < n) sp[j] = A[j];
            sp[NMAX] = b;
          }
        }
        HCX_WAVE_SYNC();
        rp = sp[k];
        if (more) next = sp[k + 1];
        HCX_WAVE_SYNC();
      };
      publish();
      // while the row is on its way: is the pivot the only one of its key?
      if constexpr (sizeof(T) == 8) {
        if (__builtin_expect(pivot_open(own, key, part, searches), 0)) {
          // the key's pivot against the others that share its bits: nothing
          // changes where they are equal (ties go to the first row)
          const double mag = cabs1(A[k]);
          const bool near = row && label >= k && same_upper(own, key);
          double top;
          if constexpr (GC > 0) {
            top = lane_read(mag, g.gbase + __builtin_ctzll(__ballot(piv) >> g.gbase));
          } else {
            double* const w = reinterpret_cast<double*>(&keys[k % kKeyWords]);
            if (piv && g.s == 0) *w = mag;
            HCX_WAVE_SYNC();
            top = *w;
            HCX_WAVE_SYNC();
          }
          bool zero = top == 0.0;
          if (__ballot(near && mag > top) & part) {
            const unsigned long long rest = largest(k, near, pivot_rest(mag, label));
            blabel = 31 - (int)((unsigned int)rest & 31u);
            zero = key < 32u && rest << 1 < 64u;
            piv = row && label == blabel;
            publish();
          }
          singular = singular || zero;
        }
      }
      if (piv) own_rinv = rinv;
      if constexpr (kSplit) {
        HCX_WAVE_SYNC();
        if (piv) {
#pragma unroll
          for (int j = k + 2; j < NMAX; ++j)
            if ((j & ~3) < n) sp[j] = A[j];
          sp[NMAX] = b;
        }
        HCX_WAVE_SYNC();
      }
      label = piv ? k : (label == k ? blabel : label);
      const bool upd = row && !piv;
      cx<T> l = cmul_fused(A[k], rp);
      l = cmk<T>(upd ? l.re : T(0), upd ? l.im : T(0));
      if (more) {
        if (GC == 0 && (k + 1) % kKeyWords == 0) clear_keys(keys, g, row);
        A[k + 1] = cfnms(A[k + 1], l, next);
        search(k + 1);
      }
#pragma unroll
      for (int j = k + 2; j < NMAX; ++j)
        if ((j & ~3) < n) A[j] = cfnms(A[j], l, sp[j]);
      b = cfnms(b, l, sp[NMAX]);
      HCX_WAVE_SYNC();
    }
  }
  const cx<T> xi = cmul_fused(b, own_rinv);
  if (row) sp[label] = xi;
  HCX_WAVE_SYNC();
  cx<T> sol = row ? sp[g.gl] : cmk<T>(T(0), T(0));
  HCX_WAVE_SYNC();
  if (singular) sol = cmk<T>(T(NAN), T(NAN));
  return sol;
}

// ------------------------------------------------------------ solve of R replicas
// One level of the reduce-scatter over the replicas: entries 2 i and 2 i + 1 of
// V, partial sums in this replica and its partner (lane src), become the sum
// of one of them, the odd one where `odd`.
template <int N>
__device__ __forceinline__ void scatter_level(const cx<double> (&V)[N], cx<double> (&W)[(N + 1) / 2], bool odd,
                                              int src) {
#pragma unroll
  for (int i = 0; i < (N + 1) / 2; ++i) {
    const cx<double> a = V[2 * i], b = 2 * i + 1 < N ? V[2 * i + 1 < N ? 2 * i + 1 : 0] : cmk<double>(0, 0);
    const cx<double> keep = odd ? b : a, send = odd ? a : b;
    W[i] = cmk<double>(keep.re + __shfl(send.re, src), keep.im + __shfl(send.im, src));
  }
}
// Partial sums V of a row's entries in the R replicas of a group -> B[i] = the
// sum of entry R i + s in replica s (the same additions as a butterfly that
// leaves every sum in every replica, level by level, a half of them each).
template <int R, int N>
__device__ __forceinline__ void reduce_scatter(const cx<double> (&V)[N], cx<double> (&B)[(N + R - 1) / R],
                                               const Group& g, int lane) {
  const int w = lane - g.s * g.G;  // this row's lane in replica 0
  cx<double> a[(N + 1) / 2];
  scatter_level(V, a, (g.s & 1) != 0, (w + (g.s ^ 1) * g.G) & 63);
  if constexpr (R == 2) {
#pragma unroll
    for (int i = 0; i < (N + 1) / 2; ++i) B[i] = a[i];
  } else {
    cx<double> b[(N + 3) / 4];
    scatter_level(a, b, (g.s & 2) != 0, (w + (g.s ^ 2) * g.G) & 63);
    if constexpr (R == 4) {
#pragma unroll
      for (int i = 0; i < (N + 3) / 4; ++i) B[i] = b[i];
    } else {
      scatter_level(b, B, (g.s & 4) != 0, (w + (g.s ^ 4) * g.G) & 63);
    }
  }
}

// Bytes of a group's LDS beyond the region of one replica: the column of the
// step in every replica, and the pivot row.
constexpr int split_bytes(int nmax, int G, int R) { return R > 1 ? 16 * (R * G + (nmax + R) / R * R) : 0; }

// group_lu_solve of a group of R replicas with the columns dealt out: replica
// s holds columns s, s + R, ... of its rows, the right-hand side as column
// NMAX.  Every replica does only its columns' updates (1 / R of the row
// broadcast and of the arithmetic), which the replicas would otherwise repeat;
// the step's column, which every row's multiplier comes from, goes to the
// other replicas through LDS while the pivot search is under way.  The same
// operations on every entry as in group_lu_solve.  cols: R * G slots, prow:
// the pivot row.
// Bound by the chain of n steps (a search of two LDS round trips, the row, a
// reciprocal), no longer by the row: one path of n = 12, R = 4: 2.82 -> 2.57 ms,
// 8 paths of n = 3, R = 8: 282 -> 261 us, n = 16, R = 2: 5.80 -> 5.24 ms.  R is a
// template argument, as the number of columns a lane holds has to be: with the
// launch's R the instances spilled (n = 16: 6.99 ms).
template <int NMAX, int R, int NC>
__device__ __forceinline__ cx<double> group_solve_split(cx<double> (&B)[NC], const Group& g, int n, bool row,
                                                        cx<double>* sp, unsigned long long* keys, cx<double>* cols,
                                                        cx<double>* prow, bool act, bool& singular) {
  static_assert(NC == (NMAX + R) / R, "columns 0..NMAX in R replicas");
  const unsigned long long part = __ballot(act);
  const int searches = g.G == 1 ? -1 : __popcll(__ballot(act && g.gl == 0 && g.s == 0));
  int label = g.gl;
  cx<double> own_rinv = cmk<double>(0, 0);
  singular = false;
  constexpr int kXWords = 2 * (NMAX + 2);
  unsigned long long* const no_key = keys - kXWords + (g.gl + g.s * g.G) % kXWords;
  cx<double>* const mine = prow + g.s;
  clear_keys(keys, g, row);
  HCX_WAVE_SYNC();
  unsigned int key = 0, own = 0;
  cx<double> ck = cmk<double>(0, 0);
  auto search = [&](int k) {
    const int so = k % R, io = k / R;
    if (g.in_grp) cols[g.s * g.G + g.gl] = B[io];
    const bool cand = row && label >= k && g.s == so;
    own = cand ? pivot_key(cabs1(B[io]), label) : 0u;
    __hip_atomic_fetch_max(reinterpret_cast<key32*>(cand ? &keys[k % kKeyWords] : no_key), own, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WAVEFRONT);
    HCX_WAVE_SYNC();
    key = *reinterpret_cast<key32*>(&keys[k % kKeyWords]);
    ck = cols[so * g.G + g.gl];
    HCX_WAVE_SYNC();
  };
  search(0);
#pragma unroll
  for (int k = 0; k < NMAX; ++k) {
    if (k < n) {
      const int so = k % R, io = k / R;
      cx<double> rinv = crecip(B[io]);  // the pivot's in replica so
      asm volatile("" : "+v"(rinv.re), "+v"(rinv.im));
      int blabel = 31 - (int)(key & 31u);
      bool piv = row && label == blabel;
      const bool more = k + 1 < NMAX && k + 1 < n;
      cx<double> rp, next = cmk<double>(0, 0);
      auto publish = [&]() {
        if (piv) {
#pragma unroll
          for (int i = io; i < NC; ++i) {
            cx<double> v = B[i];
            if (i == io) v = cmk<double>(g.s == so ? rinv.re : v.re, g.s == so ? rinv.im : v.im);
            if (R * i < n || i == NMAX / R) mine[R * i] = v;
          }
        }
        HCX_WAVE_SYNC();
        rp = prow[k];
        if (more) next = mine[R * ((k + 1) / R)];
        HCX_WAVE_SYNC();
      };
      publish();
      if (__builtin_expect(pivot_open(own, key, part, searches), 0)) {
        const double mag = cabs1(B[io]);
        const bool near = row && label >= k && g.s == so && same_upper(own, key);
        double* const w = reinterpret_cast<double*>(&keys[k % kKeyWords]);
        if (piv && g.s == so) *w = mag;
        HCX_WAVE_SYNC();
        const double top = *w;
        HCX_WAVE_SYNC();
        bool zero = top == 0.0;
        if (__ballot(near && mag > top) & part) {
          __hip_atomic_fetch_max(reinterpret_cast<key64*>(near ? &keys[k % kKeyWords] : no_key),
                                 near ? pivot_rest(mag, label) : 0ull, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_WAVEFRONT);
          HCX_WAVE_SYNC();
          const unsigned long long rest = *reinterpret_cast<key64*>(&keys[k % kKeyWords]);
          blabel = 31 - (int)((unsigned int)rest & 31u);
          zero = key < 32u && rest << 1 < 64u;
          piv = row && label == blabel;
          HCX_WAVE_SYNC();
          publish();
        }
        singular = singular || zero;
      }
      label = piv ? k : (label == k ? blabel : label);
      own_rinv = cmk<double>(piv ? rp.re : own_rinv.re, piv ? rp.im : own_rinv.im);
      const bool upd = row && !piv;
      cx<double> l = cmul_fused(ck, rp);
      l = cmk<double>(upd ? l.re : 0.0, upd ? l.im : 0.0);
      if (more) {
        if ((k + 1) % kKeyWords == 0) clear_keys(keys, g, row);
        B[(k + 1) / R] = cfnms(B[(k + 1) / R], l, next);
        search(k + 1);
      }
#pragma unroll
      for (int i = io; i < NC; ++i)
        if (i != (k + 1) / R || !more)
          if (R * i < n || i == NMAX / R) B[i] = cfnms(B[i], l, mine[R * i]);
      HCX_WAVE_SYNC();
    }
  }
  const cx<double> xi = cmul_fused(B[NMAX / R], own_rinv);
  if (row && g.s == NMAX % R) sp[label] = xi;
  HCX_WAVE_SYNC();
  cx<double> sol = row ? sp[g.gl] : cmk<double>(0, 0);
  HCX_WAVE_SYNC();
  if (singular) sol = cmk<double>(NAN, NAN);
  return sol;
}

// Copies a segment's compact term tables to the start of the dynamic LDS.
// Every wave of the block takes part (one copy per block) and the block
// barrier orders every wave's table reads after the copy; blocks of several
// waves run one segment only, so each wave reaches the barrier once.
__device__ __forceinline__ const void* stage_tables(const Seg& S, unsigned char* smem) {
  uint32_t* d = reinterpret_cast<uint32_t*>(smem);
  for (int i = (int)threadIdx.x; i < S.tab_words; i += (int)blockDim.x) d[i] = S.ctab[i];
  __syncthreads();
  return d;
}

// The full Term records of the generic instances (dH/dx streams, then dH/dt)
// copied into LDS by the block's waves; for launches of few paths (latency
// bound: no other waves hide the global latency of the evaluation's record
// loads).  Same barrier rule as stage_tables.
__device__ __forceinline__ const Term* stage_terms(const Seg& S, int n, unsigned char* smem) {
  uint4* d = reinterpret_cast<uint4*>(smem);
  const int nhx = S.hx_recs, nht = S.htT * n;
  const uint4* hx = reinterpret_cast<const uint4*>(S.hx);
  const uint4* ht = reinterpret_cast<const uint4*>(S.ht);
  for (int i = (int)threadIdx.x; i < nhx; i += (int)blockDim.x) d[i] = hx[i];
  for (int i = (int)threadIdx.x; i < nht; i += (int)blockDim.x) d[nhx + i] = ht[i];
  __syncthreads();
  return reinterpret_cast<const Term*>(d);
}

// Per-group view of the LDS region: x / pivot row, pivot keys, coefficients.
// x (read by the evaluation) and the pivot-row buffer (written by the LU that
// follows it) are never live at the same time, so they share the first
// NMAX + 1 slots (one more holds the evaluation's constant 0); group_lu_solve
// starts with a wave-scope fence that keeps the evaluation's reads before its
// writes.  KEYS: the instance searches
// pivots through LDS (no DPP groups).
constexpr int key_bytes(bool keys) { return keys ? 8 * kKeyWords : 0; }
template <int NMAX, bool KEYS>
struct Lds {
  unsigned char* base;
  __device__ cx<double>* x64() const { return reinterpret_cast<cx<double>*>(base); }
  __device__ cx<double>* piv64() const { return x64(); }
  __device__ unsigned long long* keys() const { return reinterpret_cast<unsigned long long*>(x64() + (NMAX + 2)); }
  __device__ unsigned char* coef() const { return base + 16 * (NMAX + 2) + key_bytes(KEYS); }
  template <class T>
  __device__ cx<T>* x() const { return reinterpret_cast<cx<T>*>(base); }
  template <class T>
  __device__ cx<T>* piv() const { return reinterpret_cast<cx<T>*>(piv64()); }
};

// Outputs of a finished path.
template <class SegT>
__device__ __forceinline__ void store_path(const SegT& S, long long path, int inst, int n, bool row, const Group& g,
                                           cx<double> x, uint32_t fl, int nsteps, int nnewt, int nref, double t,
                                           double dt, double resid) {
  const SegOut* O = S.out;
  double2* roots = O->roots;
  const int rstride = O->roots_stride;
  if (row && g.s == 0) roots[(size_t)path * rstride + g.gl] = make_double2(x.re, x.im);
  if (g.gl == 0 && g.s == 0) {
    if (rstride > n) roots[(size_t)path * rstride + n] = make_double2(1.0, 0.0);
    if (O->flags) O->flags[path] = fl;
    if (O->steps) O->steps[path] = nsteps;
    if (O->newton) O->newton[path] = nnewt;
    if (O->refine) O->refine[path] = nref;
    if (O->tfin) O->tfin[path] = t;
    if (O->dtfin) O->dtfin[path] = dt;
    if (O->resid) O->resid[path] = resid;
    if (O->conv8) O->conv8[path] = (fl & HCX_FLAG_TRACKED) ? 1 : 0;
    if (O->inf8) O->inf8[path] = (fl & HCX_FLAG_INFINITY) ? 1 : 0;
    if (O->debug) O->debug[path] = (fl & HCX_FLAG_TRACKED) ? make_double2(1.0, 0.0) : make_double2(t, dt);
    if (O->inst_left) {
      const int left = atomicSub(&O->inst_left[inst], 1);
      if (left == 1 && O->inst_done) O->inst_done[inst] = wall_clock64();
    } else if (O->inst_done && S.plist) {
      atomicMax(&O->inst_done[inst], (unsigned long long)wall_clock64());
    }
  }
}

}  // namespace dev

using namespace dev;

// Phases of a lane group in the path loops.
enum : int {
  kPhIdle = 0,
  kPhLoop,     // at the loop top of the step loop (…4pts.cu:116)
  kPhStage0,   // RK4 stages 0..3 (…4pts.cu:139-183)
  kPhStage1,
  kPhStage2,
  kPhStage3,
  kPhNewton,   // corrector iteration at the new t (…4pts.cu:189-223)
  kPhRefine,   // refinement iteration on H(x, 1)
  kPhResid,    // residual H(x, 1) of the refined root
  kPhOut,      // outputs pending
};


// One evaluation of the mixed loop, at FP32 or FP64: the Jacobian's row into A,
// the row of H or dH/dt (its coefficients at rhs) returned.
template <class T, int NMAX, int DEG, bool LT, int NB, class SegT>
__device__ __forceinline__ cx<T> eval_system(const SegT& S, int n, int gle, const unsigned char* xb,
                                             const unsigned char* cb, const unsigned char* rhs,
                                             const unsigned char* lt, cx<T> (&A)[NMAX]) {
  if (LT || lt) {
    constexpr int HQ = (NMAX <= 6 && sizeof(T) == 8) || DEG > 4 ? 2 : 4;
    eval_jac_blocks<NMAX, DEG, (DEG > 4 ? 2 : NB), 0, !LT && sizeof(T) == 4, T>(S, n, lt + gle * StreamRec<DEG>::kJ, 0,
                                                                              xb, cb, A);
    return eval_rhs_stream<DEG, false, HQ, (NMAX > 6), T>(S, n, gle, xb, rhs, rhs, nullptr, false, lt, 0, 1);
  }
  if constexpr (!LT) {
    const cx<T>* const sx = reinterpret_cast<const cx<T>*>(xb);
    eval_jac_terms<NMAX, DEG, T>(S, n, gle, sx, reinterpret_cast<const cx<T>*>(cb), A, nullptr, 0, 1);
    return eval_rhs_terms<DEG, false, T>(S, n, gle, sx, reinterpret_cast<const cx<T>*>(rhs), nullptr, false, nullptr, 0,
                                         1);
  }
  return cmk<T>(0, 0);
}

// Mixed-precision lane-group path loop: FP32 RK4 predictor (Jacobian, dH/dt
// and solve of the four stages), FP64 Newton corrector (FP32 before the end
// zone when o.newton32), FP64 refinement; a path that ends without a refined
// root is re-tracked from t = 0 entirely in FP64 (escalation) by the FP64 pass
// after the launch, which keeps the FP64 predictor out of the kernel and with
// it the registers of a second predictor.
// The wave alternates between the predictor of every group that steps and
// FP64 iterations.  An FP64 iteration serves every group that has one to do: the
// corrector, the refinement and the final residual.  The FP64 turn ends when no
// group corrects any more; a group that refines goes on in the next turn, beside
// the others' correctors, so that no group waits for another's refinement.
// Streams, staging and rounds are those of the FP64 loop, at FP32 on half the
// bytes (hcx_eval.hpp); the FP32 c(t) and dc/dt of the predictor and the FP64 c(t)
// share the coefficient area.
// NB: Jacobian columns evaluated together (twice as many in FP32 were no
// faster: the rounds of a block are its longest column's).
// Bound by latency at the 7 waves per CU that its LDS allows (VALU 57% and LDS
// 61% busy).  n = 12, 240 coefficients, degrees 2 and 3, 512 x 1024
// paths: 159.5 -> 150.3 ms over the padded tables, 137.4 ms with 7 waves for 6,
// 135.1 with every gather of a round requested up front.
template <int NMAX, int DEG, bool EXACT, int NB = (NMAX <= 6 ? 3 : (NMAX <= 16 ? 4 : 6))>
__device__ __forceinline__ void run_segment_mixed(const Launch& LN, int si, unsigned char* smem, int lane) {
  Seg S = LN.seg[si];
  constexpr int GE = exact_lanes(NMAX);
  if (EXACT) {
    S.n = NMAX;
    S.G = GE;
  }
  constexpr int GC = (EXACT && is_pow2(GE)) ? GE : 0;
  const KOpts* const opts_arg = launch_opts();
  const KSeg* const seg_arg = launch_seg(si);
  int iter = 0;
  const Group g = make_group(S.G, lane);
  const int n = S.n;
  const bool row = g.in_grp && g.gl < n;
  const int gle = row ? g.gl : 0;
  constexpr bool LT = EXACT && (NMAX <= 16 || DEG <= 2);
  const unsigned char* lt = nullptr;
  if constexpr (LT) {
    lt = static_cast<const unsigned char*>(stage_tables(S, smem));
  } else if constexpr (!EXACT) {
    if (LN.tab_lds > 0) lt = static_cast<const unsigned char*>(stage_tables(S, smem));
  }
  constexpr int SQ = NMAX <= 16 ? 4 : 2;  // coefficients in flight per lane while staging
  constexpr bool SL = LT && NMAX <= 16;
  const int wv = (int)threadIdx.x >> 6;  // wave of the block
  Lds<NMAX, GC == 0> L{smem + LN.tab_lds + ((size_t)wv * g.gpw + (g.in_grp ? g.grp : 0)) * S.lds_group};
  unsigned char* const xb = L.base;
  unsigned char* const cb = L.coef();
  const int head = (int)(cb - xb);
  const unsigned char* const db = cb + S.nslot * 8;  // dc/dt (FP32)
  const double2 *hxi = S.chx, *hti = S.cht;

  long long path = -1;
  int inst = 0, root = 0;
  double t = 0.0, dt = 0.0, tst = -1.0, resid = 0.0;  // tst: t of the FP64 c(t) in LDS
  int cnt = 0, nsteps = 0, asteps = 0, nnewt = 0, nref = 0, nit = 0;
  bool ez = false, conv = false, sing_any = false;
  int ph = kPhIdle;
  uint32_t fl = 0;
  bool exhausted = !g.in_grp;
  long long static_path = ((long long)((int)blockIdx.x - LN.first_block[si]) * LN.wpb + wv) * g.gpw + g.grp;
  double ts = 0.0;
  cx<double> x = cmk<double>(0, 0), xl = x;

  for (;;) {
    const KOpts& o = *iteration_view(opts_arg, iter);
    const KSeg& Sk = *iteration_view(seg_arg, iter);
    ++iter;
    // ------------------------------------------------ refill idle groups
    const bool want = ph == kPhIdle && !exhausted;
    if (__any(want)) {
      long long p;
      if (LN.persistent) {
        unsigned int q = 0;
        if (want && g.gl == 0) {
          q = atomicAdd(Sk.counter, 1u);
          // path-list launch
          if (Sk.plist) q = q < *Sk.plist_count ? (unsigned int)Sk.plist[q] : 0xffffffffu;
        }
        p = (long long)(unsigned int)lane_read((int)q, g.gbase);
        if (p == 0xffffffffll) p = -1;
      } else {
        p = static_path;
      }
      if (want) {
        if (p < 0 || p >= Sk.P) {
          exhausted = true;
        } else {
          path = p;
          inst = (int)(p / Sk.K);
          root = (int)(p - (long long)inst * Sk.K);
          hxi = Sk.chx + (size_t)inst * (Sk.C + 1) * (Sk.M + 1);
          hti = Sk.cht + (size_t)inst * (Sk.C + 1) * Sk.M;
          nsteps = asteps = nnewt = nref = cnt = 0;
          fl = Sk.plist ? HCX_FLAG_ESCALATED : 0u;
          t = 0.0;
          dt = o.dt0;
          ez = false;
          tst = -1.0;
          resid = 0.0;
          if (row) {
            const double2 v = Sk.start[(size_t)root * Sk.start_stride + g.gl];
            x = cmk<double>(v.x, v.y);
          } else {
            x = cmk<double>(0, 0);
          }
          xl = x;
          ph = kPhLoop;
          if (!LN.persistent) exhausted = true;
        }
      }
    }
    if (!__any(ph != kPhIdle)) break;

    // ------------------------------------------------ loop top (:116-131)
    bool fin = false, stepping = false;
    if (ph == kPhLoop) {
      if (!(t < 1.0 && 1.0 - t > o.t_tol)) {
        fl |= HCX_FLAG_TRACKED;
        fin = true;
      } else if (asteps > o.max_steps) {
        fl |= HCX_FLAG_BUDGET;
        fin = true;
      } else {
        // end zone and step clamp
        if (!ez && fabs(1.0 - t) <= o.ez_enter) ez = true;
        if (ez) {
          if (dt > fabs(1.0 - t)) dt = fabs(1.0 - t);
        } else if (dt > fabs(o.ez_land - t)) {
          dt = fabs(o.ez_land - t);
        }
        ts = t;
        stepping = true;
      }
    }
    if (__any(fin)) {
      // the reference's real test on the tracked root, before refinement
      // (Evaluations.cpp:96-104: converged and every |Im x_i| <= 1e-4)
      double imt = (fin && row) ? fabs(x.im) : 0.0;
      if (imt != imt) imt = INFINITY;
      imt = group_max(imt, g);
      if (fin) {
        if ((fl & HCX_FLAG_TRACKED) && imt <= o.real_ref_tol) fl |= HCX_FLAG_REAL_REF;
        if ((fl & HCX_FLAG_TRACKED) && o.refine_iters > 0) {
          ph = kPhRefine;
          nit = 0;
          conv = false;
          sing_any = false;
        } else {
          ph = kPhOut;
        }
      }
    }

    // step control (:225-249) of a corrected step
    auto control = [&](bool ok, bool inf) {
      ++nsteps;
      ++asteps;
      ph = kPhLoop;
      if (inf) {
        fl |= HCX_FLAG_INFINITY;
        ph = kPhOut;
      } else if (!ok) {
        dt *= 0.5;
        x = xl;
        t = ts;
        cnt = 0;
        if (dt < o.dt_min) {
          fl |= HCX_FLAG_MINSTEP;
          ph = kPhOut;
        }
      } else {
        ++cnt;
        xl = x;
        if (cnt >= o.incr) {
          cnt = 0;
          dt *= 2.0;
        }
      }
    };

    // ------------------------------------------------ FP32 predictor
    if (__any(stepping)) {
      // RK4 (:139-183): stages at (x0, t), (x0 + h k1, t + h),
      // (x0 + h k2, t + h), (x0 + dt k3, t + dt)
      const double h = 0.5 * dt;
      cx<double> acc = cmk<double>(0, 0), kp = acc;
      cx<float>* const sx = L.template x<float>();
#pragma unroll 1
      for (int st = 0; st < 4; ++st) {
        const double a = st == 0 ? 0.0 : (st == 3 ? dt : h);
        // order 1: dc/dt does not depend on t, but the FP64 c(t) of the last
        // corrector lies over it
        if (stepping && st != 2)
          stage_coeffs<SL, SQ, float>(Sk, g, hxi, hti, ts + a, xb + head / 2, head, Sk.nslot * 8, st == 0 || Sk.M > 1,
                                      lt);
        const cx<double> xs = cmk<double>(xl.re + a * kp.re, xl.im + a * kp.im);
        publish_x<float>(sx, xs, g, n, stepping, row);
        HCX_WAVE_SYNC();
        cx<float> A[NMAX];
        const cx<float> bt = eval_system<float, NMAX, DEG, LT, NB>(Sk, n, gle, xb, cb, db, lt, A);
        bool sing;
        const cx<float> k = group_lu_solve<NMAX, GC, float>(A, cmk<float>(-bt.re, -bt.im), g, n, row, stepping,
                                                            L.template piv<float>(), L.keys(), sing);
        kp = ccast<double>(k);
        const double w = (st == 1 || st == 2) ? 2.0 : 1.0;
        acc = cmk<double>(acc.re + w * kp.re, acc.im + w * kp.im);
      }
      if (stepping) {
        const double f = dt * (1.0 / 6.0);
        x = cmk<double>(xl.re + f * acc.re, xl.im + f * acc.im);
        t = ts + dt;
        ph = kPhNewton;
        nit = 0;
        tst = -1.0;
      }
      // FP32 corrector before the end zone (o.newton32), on stage 3's c(t + dt)
      bool run = stepping && !ez && o.newton32;
      if (__any(run)) {
        const bool run32 = run;
        bool ok = false, inf = false;
        for (int it = 0; it < o.max_corr; ++it) {
          if (!__any(run)) break;
          publish_x<float>(sx, x, g, n, run, row);
          HCX_WAVE_SYNC();
          cx<float> A[NMAX];
          const cx<float> hv = eval_system<float, NMAX, DEG, LT, NB>(Sk, n, gle, xb, cb, cb, lt, A);
          bool sing;
          const cx<float> d =
              group_lu_solve<NMAX, GC, float>(A, hv, g, n, row, run, L.template piv<float>(), L.keys(), sing);
          if (run && row) x = csub(x, ccast<double>(d));
          double s1 = row ? (double)cnorm2(d) : 0.0, s2 = row ? cnorm2(x) : 0.0;
          group_sum2<NMAX, GC, true>(s1, s2, g, n, row, lane, L.piv64());
          if (run) {
            ++nnewt;
            ok = s1 < o.corr_tol * s2;
            inf = s2 > o.inf_tol;
            if (ok || inf) run = false;
          }
        }
        if (run32) control(ok, inf);
        HCX_WAVE_SYNC();
      }
    }

    // ------------------------------------------------ FP64 iterations
    for (;;) {
      const int pe = ph;
      const bool act = pe == kPhNewton || pe == kPhRefine || pe == kPhResid;
      if (!__any(act)) break;
      const double te = pe == kPhNewton ? t : 1.0;
      if (act && te != tst) {
        stage_coeffs<SL, SQ, double>(Sk, g, hxi, hti, te, xb, head, 0, false, lt);
        tst = te;
      }
      cx<double>* const sx = L.x64();
      publish_x<double>(sx, x, g, n, act, row);
      HCX_WAVE_SYNC();
      cx<double> A[NMAX];
      const cx<double> r = eval_system<double, NMAX, DEG, LT, NB>(Sk, n, gle, xb, cb, cb, lt, A);
      bool sing;
      const cx<double> d = group_lu_solve<NMAX, GC, double>(A, r, g, n, row, act, L.piv64(), L.keys(), sing);
      const bool nr = pe == kPhNewton || pe == kPhRefine;
      if (nr && row) x = csub(x, d);
      double s1 = (nr && row) ? cnorm2(d) : 0.0, s2 = (nr && row) ? cnorm2(x) : 0.0;
      group_sum2<NMAX, GC, true>(s1, s2, g, n, row, lane, L.piv64());
      if (pe == kPhNewton) {
        ++nnewt;
        ++nit;
        const bool ok = s1 < o.corr_tol * s2, inf = s2 > o.inf_tol;
        if (ok || inf || nit >= o.max_corr) control(ok, inf);
      } else if (pe == kPhRefine) {
        ++nref;
        ++nit;
        sing_any = sing;
        bool stop = false;
        if (!(s2 < o.inf_tol)) {
          stop = true;
        } else if (sqrt(s1) <= o.refine_tol * fmax(1.0, sqrt(s2))) {
          conv = true;
          stop = true;
        }
        if (stop || nit >= o.refine_iters) ph = kPhResid;
      }
      // residual max_i |H_i(x, 1)| of the refined root (r = H at x)
      const bool rz = pe == kPhResid;
      if (__any(rz)) {
        double rr = (rz && row) ? sqrt(cnorm2(r)) : 0.0;
        if (rr != rr) rr = INFINITY;
        rr = group_max(rr, g);
        double im = (rz && row) ? fabs(x.im) : 0.0;
        if (im != im) im = INFINITY;
        im = group_max(im, g);
        if (rz) {
          resid = rr;
          if (conv) fl |= HCX_FLAG_REFINED;
          if (conv && im <= o.real_tol) fl |= HCX_FLAG_REAL;
          if (sing_any) fl |= HCX_FLAG_SINGULAR;
          ph = kPhOut;
        }
      }
      HCX_WAVE_SYNC();
      if (!__any(ph == kPhNewton)) break;
    }

    // ------------------------------------------------ outputs
    const bool out = ph == kPhOut;
    if (__any(out) && out) {
      store_path(Sk, path, inst, n, row, g, x, fl, nsteps, nnewt, nref, t, dt, resid);
      ph = kPhIdle;
      path = -1;
    }
  }
}

// FP64 lane-group path loop in uniform micro-steps.  Every iteration of the
// wave performs ONE evaluation (Jacobian rows and a right-hand side) and ONE
// group solve for every active group, whatever each group's path is doing:
// an RK4 stage, a corrector iteration, a refinement iteration or the final
// residual.  A group that leaves a phase (a corrector that converges after
// one iteration, a path that ends) takes its next micro-step in the next
// iteration, so no group waits for the slowest group of its wave to finish a
// phase.  Each path's sequence of operations and results are those of the
// step loop (…4pts.cu:115-254) and of the refinement: only the interleaving
// of the groups of a wave changes.  c(t) is staged in LDS only when the
// group's evaluation point moves (RK4 stages 0, 1 and 3; the corrector
// reuses stage 3's c(t + dt)).
// REP: 0: the throughput loop; else the latency instance (launches of few
// paths, two waves per SIMD at most): 2, 4 or 8 replicas per path, which share
// the evaluation's terms and the solve's columns, or (1) Seg::R of them, which
// share the terms.
// DEAL: the replicas share the columns in the evaluation as well: each sums its
// own whole, in the order of one replica, and all of them the right-hand side.
// 142 paths of each of 64 instances of n = 9, R = 2: 3.46 -> 3.03 ms.
// NB: Jacobian columns evaluated together (as the register budget allows).
template <int NMAX, int DEG, bool EXACT, int REP, int NB = (NMAX <= 6 ? 3 : (NMAX <= 16 ? 4 : 6)), bool DEAL = false>
__device__ __forceinline__ void run_segment_fp64(const Launch& LN, int si, unsigned char* smem, int lane) {
  Seg S = LN.seg[si];
  constexpr int GE = exact_lanes(NMAX);
  if (EXACT) {
    S.n = NMAX;
    S.G = GE;
  }
  constexpr int GC = (EXACT && is_pow2(GE)) ? GE : 0;
  const KOpts* const opts_arg = launch_opts();
  const KSeg* const seg_arg = launch_seg(si);
  int iter = 0;
  const Group g = make_group(S.G, lane, REP > 1 ? REP : (REP ? S.R : 1));
  if constexpr (REP == 0) {
    // a list with too few paths for this wave (persistent launches of one-wave
    // blocks; each segment's first waves cover its list)
    if (S.plist) {
      const int rel = (int)blockIdx.x - LN.first_block[si], paths = (int)*S.plist_count;
      if (rel >= (paths + g.gpw - 1) / g.gpw) return;
    }
  }
  // the replica's terms of each sum
  const int k0 = REP && !DEAL ? g.s : 0, ks = DEAL ? 1 : (REP > 1 ? REP : (REP ? g.R : 1));
  const int n = S.n;
  const bool row = g.in_grp && g.gl < n;
  const int gle = row ? g.gl : 0;
  constexpr bool LT = EXACT && (NMAX <= 16 || DEG <= 2);
  // The compact streams in LDS: always (LT), or in a generic instance where
  // the launch found room for them; else the full Term records in global
  // memory, or (generic latency instance) in LDS.  tab_lds holds the bytes.
  const unsigned char* lt = nullptr;
  const Term* tl = nullptr;
  if constexpr (LT) {
    lt = static_cast<const unsigned char*>(stage_tables(S, smem));
  } else if constexpr (!EXACT) {
    if (LN.tab_lds > 0 && S.ctab) {
      lt = static_cast<const unsigned char*>(stage_tables(S, smem));
    } else if constexpr (REP) {
      if (LN.tab_lds > 0) tl = stage_terms(S, n, smem);
    }
  }
  // coefficients in flight per lane while staging (order 1)
  constexpr int SQ = EXACT && NMAX <= 16 ? 4 : 2;
  const int wv = (int)threadIdx.x >> 6;  // wave of the block
  Lds<NMAX, GC == 0 || (REP > 0)> L{smem + LN.tab_lds + ((size_t)wv * g.gpw + (g.in_grp ? g.grp : 0)) * S.lds_group};
  cx<double>* sx = L.x64();
  unsigned char* const xb = L.base;
  unsigned char* const cb = L.coef();
  unsigned char* const db = cb + S.nslot * 16;  // dc/dt, when in LDS
  // the split solve's columns and pivot row (latency instances: dc/dt is in LDS)
  cx<double>* const cols = reinterpret_cast<cx<double>*>(db + S.nslot * 16);
  // the path's instance tables
  const double2 *hxi = S.chx, *hti = S.cht;
  // dc/dt of the RK4 stages: constant (M = 1) -> read from the instance's
  // table in global memory (half the group's LDS), unless the launch stages
  // it in LDS (dot_lds: launches of few paths, and every latency instance);
  // M > 1 -> LDS
  const bool gdot = REP == 0 && S.M == 1 && !LN.dot_lds;

  long long path = -1;
  int inst = 0, root = 0;
  double t = 0.0, dt = 0.0, ts = 0.0, tst = -1.0, resid = 0.0;
  int cnt = 0, nsteps = 0, asteps = 0, nnewt = 0, nref = 0, nit = 0;
  bool ez = false, conv = false, sing_any = false;
  int ph = kPhIdle;
  uint32_t fl = 0;
  bool exhausted = !g.in_grp;
  long long static_path = ((long long)((int)blockIdx.x - LN.first_block[si]) * LN.wpb + wv) * g.gpw + g.grp;
  cx<double> x = cmk<double>(0, 0), xl = x, acc = x, kp = x;

  for (;;) {
    const KOpts& o = *iteration_view(opts_arg, iter);
    const KSeg& Sk = *iteration_view(seg_arg, iter);
    ++iter;
    // ------------------------------------------------ refill idle groups
    const bool want = ph == kPhIdle && !exhausted;
    if (__any(want)) {
      long long p;
      if (LN.persistent) {
        unsigned int q = 0;
        if (want && g.gl == 0 && g.s == 0) {
          q = atomicAdd(Sk.counter, 1u);
          if (Sk.plist) q = q < *Sk.plist_count ? (unsigned int)Sk.plist[q] : 0xffffffffu;
        }
        p = (long long)(unsigned int)lane_read((int)q, g.wbase);
        if (p == 0xffffffffll) p = -1;
      } else {
        p = static_path;
      }
      if (want) {
        if (p < 0 || p >= Sk.P) {
          exhausted = true;
        } else {
          path = p;
          inst = (int)(p / Sk.K);
          root = (int)(p - (long long)inst * Sk.K);
          hxi = Sk.chx + (size_t)inst * (Sk.C + 1) * (Sk.M + 1);
          hti = Sk.cht + (size_t)inst * (Sk.C + 1) * Sk.M;
          nsteps = asteps = nnewt = nref = cnt = 0;
          fl = Sk.plist ? HCX_FLAG_ESCALATED : 0u;
          t = 0.0;
          dt = o.dt0;
          ez = false;
          tst = -1.0;  // the LDS coefficients belong to another instance
          resid = 0.0;
          if (row) {
            const double2 v = Sk.start[(size_t)root * Sk.start_stride + g.gl];
            x = cmk<double>(v.x, v.y);
          } else {
            x = cmk<double>(0, 0);
          }
          xl = x;
          ph = kPhLoop;
          if (!LN.persistent) exhausted = true;
        }
      }
    }
    if (!__any(ph != kPhIdle)) break;

    // ------------------------------------------------ loop top (:116-131)
    bool fin = false;
    if (ph == kPhLoop) {
      if (!(t < 1.0 && 1.0 - t > o.t_tol)) {
        fl |= HCX_FLAG_TRACKED;
        fin = true;
      } else if (asteps > o.max_steps) {
        fl |= HCX_FLAG_BUDGET;
        fin = true;
      } else {
        if (!ez && fabs(1.0 - t) <= o.ez_enter) ez = true;
        if (ez) {
          if (dt > fabs(1.0 - t)) dt = fabs(1.0 - t);
        } else if (dt > fabs(o.ez_land - t)) {
          dt = fabs(o.ez_land - t);
        }
        ts = t;
        acc = cmk<double>(0, 0);
        kp = acc;
        ph = kPhStage0;
      }
    }
    if (__any(fin)) {
      // the reference's real test on the tracked root, before refinement
      // (Evaluations.cpp:96-104: converged and every |Im x_i| <= 1e-4)
      double imt = (fin && row) ? fabs(x.im) : 0.0;
      if (imt != imt) imt = INFINITY;
      imt = group_max(imt, g);
      if (fin) {
        if ((fl & HCX_FLAG_TRACKED) && imt <= o.real_ref_tol) fl |= HCX_FLAG_REAL_REF;
        if ((fl & HCX_FLAG_TRACKED) && o.refine_iters > 0) {
          ph = kPhRefine;
          nit = 0;
          conv = false;
          sing_any = false;
        } else {
          ph = kPhOut;
        }
      }
    }

    // ------------------------------------------------ one micro-step
    const int pe = ph;
    const bool stg = pe >= kPhStage0 && pe <= kPhStage3;
    const bool act = stg || pe == kPhNewton || pe == kPhRefine || pe == kPhResid;
    if (__any(act)) {
      const int k = pe - kPhStage0;
      const double a = k == 0 ? 0.0 : (k == 3 ? dt : 0.5 * dt);
      const double te = stg ? ts + a : (pe == kPhNewton ? t : 1.0);
      const cx<double> xe = stg ? cmk<double>(xl.re + a * kp.re, xl.im + a * kp.im) : x;
      const bool restage = act && te != tst;
      if (restage) {
        // order 1: dc/dt does not depend on t, once per path is enough
        const bool dot = !gdot && (Sk.M > 1 || tst < 0.0);
        stage_coeffs<LT && NMAX <= 16, SQ, double>(Sk, g, hxi, hti, te, xb, (int)(cb - xb), (int)(db - cb), dot, lt);
        tst = te;
      }
      publish_x<double>(sx, xe, g, n, act, row);
      HCX_WAVE_SYNC();
      constexpr int NC = REP > 1 ? (NMAX + REP) / REP : 1;  // columns of a replica (the right-hand side's included)
      cx<double> A[NMAX], B[NC];
      cx<double> r;
      if (DEAL || LT || (!EXACT && lt)) {
        constexpr bool kPin = REP > 0 || NMAX > 6;
        if constexpr (REP) {
          if constexpr (DEAL)
            eval_jac_dealt<NMAX, DEG, REP, NC>(Sk, n, gle, g.s, xb, cb, B, lt);
          else
            eval_jac_rounds<NMAX, DEG>(Sk, n, gle, xb, cb, A, lt, k0, ks);
          if (DEG > 4 || Sk.htT <= 2 * ks)
            r = eval_rhs_stream<DEG, false, 2, kPin, double>(Sk, n, gle, xb, cb, db, hti, stg, lt, k0, ks);
          else
            r = eval_rhs_stream<DEG, false, 4, kPin, double>(Sk, n, gle, xb, cb, db, hti, stg, lt, k0, ks);
        } else {
          constexpr int HQ = NMAX <= 6 || DEG > 4 ? 2 : 4;  // H terms in flight
          eval_jac_blocks<NMAX, DEG, (DEG > 4 ? 2 : NB), 0, false, double>(Sk, n, lt + gle * StreamRec<DEG>::kJ, 0, xb,
                                                                           cb, A);
          if (gdot)
            r = eval_rhs_stream<DEG, true, HQ, kPin, double>(Sk, n, gle, xb, cb, db, hti, stg, lt, k0, ks);
          else
            r = eval_rhs_stream<DEG, false, HQ, kPin, double>(Sk, n, gle, xb, cb, db, hti, stg, lt, k0, ks);
        }
      } else {
        const cx<double>* sc = reinterpret_cast<const cx<double>*>(cb);
        eval_jac_terms<NMAX, DEG, double>(Sk, n, gle, sx, sc, A, tl, k0, ks);
        if (gdot)
          r = eval_rhs_terms<DEG, true, double>(Sk, n, gle, sx, sc, hti, stg, tl, k0, ks);
        else
          r = eval_rhs_terms<DEG, false, double>(Sk, n, gle, sx, reinterpret_cast<const cx<double>*>(stg ? db : cb), hti, stg,
                                         tl, k0, ks);
      }
      bool sing;
      cx<double> d;
      if constexpr (REP > 1) {
        cx<double>& rb = B[NMAX / REP];  // (the right-hand side: in replica NMAX % REP)
        if constexpr (DEAL) {
          if (g.s == NMAX % REP) rb = stg ? cmk<double>(-r.re, -r.im) : r;
        } else {
          // each replica summed every R-th term of the row's sums
          cx<double> V[NMAX + 1];
#pragma unroll
          for (int j = 0; j < NMAX; ++j) V[j] = A[j];
          V[NMAX] = r;
          reduce_scatter<REP>(V, B, g, lane);
          r = rb;
          if (stg && g.s == NMAX % REP) rb = cmk<double>(-rb.re, -rb.im);
        }
        d = group_solve_split<NMAX, REP>(B, g, n, row, L.piv64(), L.keys(), cols, cols + REP * g.G, act, sing);
      } else {
        if constexpr (REP == 1) {
          // more replicas than the split solve deals out: a butterfly over
          // them (all sums of a level exchanged together) leaves the full
          // sums, identical in every replica (each level adds a pair of
          // partial sums, commutatively)
          for (int m = 1; m < g.R; m <<= 1) {
            const int src = (lane + ((g.s ^ m) - g.s) * g.G) & 63;
#pragma unroll
            for (int j = 0; j < NMAX; ++j) {
              if (j < n) {
                A[j].re += __shfl(A[j].re, src);
                A[j].im += __shfl(A[j].im, src);
              }
            }
            r.re += __shfl(r.re, src);
            r.im += __shfl(r.im, src);
          }
        }
        d = group_lu_solve<NMAX, GC, double>(A, stg ? cmk<double>(-r.re, -r.im) : r, g, n, row, act, L.piv64(),
                                             L.keys(), sing);
      }

      // RK4 stage: k_s = solution, accumulate k1 + 2 k2 + 2 k3 + k4
      if (stg) {
        kp = d;
        const double w = (k == 1 || k == 2) ? 2.0 : 1.0;
        acc = cmk<double>(acc.re + w * kp.re, acc.im + w * kp.im);
        if (k == 3) {
          const double f = dt * (1.0 / 6.0);
          x = cmk<double>(xl.re + f * acc.re, xl.im + f * acc.im);
          t = ts + dt;
          ph = kPhNewton;
          nit = 0;
        } else {
          ph = pe + 1;
        }
      }
      // corrector and refinement iterations: x -= d and the group norms
      const bool nr = pe == kPhNewton || pe == kPhRefine;
      if (nr && row) x = csub(x, d);
      double s1 = (nr && row) ? cnorm2(d) : 0.0, s2 = (nr && row) ? cnorm2(x) : 0.0;
      if (__any(nr)) group_sum2<NMAX, GC, false>(s1, s2, g, n, row, lane, L.template piv<double>());
      if (pe == kPhNewton) {
        ++nnewt;
        ++nit;
        const bool ok = s1 < o.corr_tol * s2, inf = s2 > o.inf_tol;
        if (ok || inf || nit >= o.max_corr) {
          // step control (:225-249)
          ++nsteps;
          ++asteps;
          if (inf) {
            fl |= HCX_FLAG_INFINITY;
            ph = kPhOut;
          } else if (!ok) {
            dt *= 0.5;
            x = xl;
            t = ts;
            cnt = 0;
            if (dt < o.dt_min) {
              fl |= HCX_FLAG_MINSTEP;
              ph = kPhOut;
            } else {
              ph = kPhLoop;
            }
          } else {
            ++cnt;
            xl = x;
            if (cnt >= o.incr) {
              cnt = 0;
              dt *= 2.0;
            }
            ph = kPhLoop;
          }
        }
      } else if (pe == kPhRefine) {
        ++nref;
        ++nit;
        sing_any = sing;
        bool stop = false;
        if (!(s2 < o.inf_tol)) {
          stop = true;
        } else if (sqrt(s1) <= o.refine_tol * fmax(1.0, sqrt(s2))) {
          conv = true;
          stop = true;
        }
        if (stop || nit >= o.refine_iters) ph = kPhResid;
      }
      // residual max_i |H_i(x, 1)| of the refined root (r = H at x)
      const bool rz = pe == kPhResid;
      if (__any(rz)) {
        // the replica that holds the right-hand side's column has the sums
        if constexpr (REP > 1 && !DEAL) r = lane_read(r, g.wbase + (NMAX % REP) * g.G + g.gl);
        double rr = (rz && row) ? sqrt(cnorm2(r)) : 0.0;
        if (rr != rr) rr = INFINITY;
        rr = group_max(rr, g);
        double im = (rz && row) ? fabs(x.im) : 0.0;
        if (im != im) im = INFINITY;
        im = group_max(im, g);
        if (rz) {
          resid = rr;
          if (conv) fl |= HCX_FLAG_REFINED;
          if (conv && im <= o.real_tol) fl |= HCX_FLAG_REAL;
          if (sing_any) fl |= HCX_FLAG_SINGULAR;
          ph = kPhOut;
        }
      }
      HCX_WAVE_SYNC();
    }

    // ------------------------------------------------ outputs
    const bool out = ph == kPhOut;
    if (__any(out) && out) {
      // replica 0 stores (the other replicas hold the same values)
      store_path(Sk, path, inst, n, row, g, x, fl, nsteps, nnewt, nref, t, dt, resid);
      ph = kPhIdle;
      path = -1;
    }
  }
}

// Register budget: the size-specialised instances up to n = 6 are compiled
// for three waves per SIMD (at most 168 VGPRs), the others up to 16 variables
// for two, which their live state fits with few spills or none.
constexpr int waves_per_simd(int nmax, bool exact) { return exact && nmax <= 6 ? 3 : (nmax <= 16 ? 2 : 1); }
// Blocks of up to 8 waves, as many as fit the CU's four SIMDs.
constexpr int block_threads(int nmax, bool exact) { return waves_per_simd(nmax, exact) > 1 ? 512 : 256; }
template <int NMAX, int DEG, int MODE, bool EXACT>
__global__ __launch_bounds__(block_threads(NMAX, EXACT)) __attribute__((amdgpu_waves_per_eu(waves_per_simd(NMAX, EXACT))))
void track_kernel(const Launch LN) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = (int)threadIdx.x & 63;
  int s = 0;
  while (s + 1 < LN.nseg && (int)blockIdx.x >= LN.first_block[s + 1]) ++s;
  for (int tried = 0; tried < LN.nseg; ++tried) {
    if constexpr (MODE == 0) {
      run_segment_fp64<NMAX, DEG, EXACT, 0>(LN, s, smem, lane);
    } else {
      run_segment_mixed<NMAX, DEG, EXACT>(LN, s, smem, lane);
    }
    if (!LN.persistent) break;
    s = s + 1 == LN.nseg ? 0 : s + 1;
  }
}

// Latency instance: FP64 launches of one segment and few paths, R replicas
// per path (1: the launch's number).
template <int NMAX, int DEG, bool EXACT, int R, bool DEAL = false>
__global__ __launch_bounds__(block_threads(NMAX, false)) __attribute__((amdgpu_waves_per_eu(waves_per_simd(NMAX, false))))
void track_kernel_rep(const Launch LN) {
  extern __shared__ __align__(16) unsigned char smem[];
  run_segment_fp64<NMAX, DEG, EXACT, R, 4, DEAL>(LN, 0, smem, (int)threadIdx.x & 63);
}

// One launch over segments of different sizes (uneven batches): segment s
// runs the size-specialised loop of its n, n in {3, 5, 6, 9, 12} (terms of
// degree <= DEG, compact tables in LDS, G = n), so a multi-type launch keeps
// the specialised code of each type instead of the generic instance; the
// kernel's registers and LDS are those of its largest member.
template <int N, int DEG, int MODE>
__device__ __forceinline__ void run_exact(const Launch& LN, int si, unsigned char* smem, int lane) {
  if constexpr (MODE == 0) {
    run_segment_fp64<N, DEG, true, 0, 2>(LN, si, smem, lane);
  } else {
    run_segment_mixed<N, DEG, true, 2>(LN, si, smem, lane);
  }
}

template <int DEG, int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void track_kernel_set(const Launch LN) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = (int)threadIdx.x & 63;
  int s = 0;
  while (s + 1 < LN.nseg && (int)blockIdx.x >= LN.first_block[s + 1]) ++s;
  for (int tried = 0; tried < LN.nseg; ++tried) {
    switch (LN.seg[s].n) {
      case 3: run_exact<3, DEG, MODE>(LN, s, smem, lane); break;
      case 5: run_exact<5, DEG, MODE>(LN, s, smem, lane); break;
      case 6: run_exact<6, DEG, MODE>(LN, s, smem, lane); break;
      case 9: run_exact<9, DEG, MODE>(LN, s, smem, lane); break;
      case 12: run_exact<12, DEG, MODE>(LN, s, smem, lane); break;
      default: break;
    }
    if (!LN.persistent) break;
    s = s + 1 == LN.nseg ? 0 : s + 1;
  }
}

using KernelFn = void (*)(const Launch);

// Kernel instances live in separate translation units (compile in parallel).
// Generic instances: any n <= NMAX and any lanes-per-path G >= n; one unit
// per (NMAX, mode, term degree) and a dispatcher per (NMAX, mode).
KernelFn kernel_g8_m0(int deg);
KernelFn kernel_g8_m1(int deg);
KernelFn kernel_g16_m0(int deg);
KernelFn kernel_g16_m1(int deg);
KernelFn kernel_g32_m0(int deg);
KernelFn kernel_g32_m1(int deg);
#define HCX_GENERIC_UNITS(G, M) \
  KernelFn kernel_g##G##_m##M##_d2(); KernelFn kernel_g##G##_m##M##_d3(); \
  KernelFn kernel_g##G##_m##M##_d4(); KernelFn kernel_g##G##_m##M##_d6();
HCX_GENERIC_UNITS(8, 0)
HCX_GENERIC_UNITS(8, 1)
HCX_GENERIC_UNITS(16, 0)
HCX_GENERIC_UNITS(16, 1)
HCX_GENERIC_UNITS(32, 0)
HCX_GENERIC_UNITS(32, 1)
#undef HCX_GENERIC_UNITS
// Size-specialised instances (n = G = N) for the problem sizes of the
// benchmark workloads and of the reference's small problems (n = 4, 8, 10),
// DEG 2 and 3; DEG 4 for n = 4, 5 in FP64 mode.
// Multi-size instances (n in {3, 5, 6, 9, 12}, DEG 2) for uneven batches.
KernelFn kernel_set_m0();
KernelFn kernel_set_m1();
KernelFn kernel_x3_m0(int deg);
KernelFn kernel_x3_m1(int deg);
KernelFn kernel_x4_m0(int deg);
KernelFn kernel_x4_m1(int deg);
KernelFn kernel_x5_m0(int deg);
KernelFn kernel_x5_m1(int deg);
KernelFn kernel_x6_m0(int deg);
KernelFn kernel_x6_m1(int deg);
KernelFn kernel_x8_m0(int deg);
KernelFn kernel_x8_m1(int deg);
KernelFn kernel_x9_m0(int deg);
KernelFn kernel_x9_m1(int deg);
KernelFn kernel_x10_m0(int deg);
KernelFn kernel_x10_m1(int deg);
KernelFn kernel_x12_m0(int deg);
KernelFn kernel_x12_m1(int deg);
KernelFn kernel_x16_m0(int deg);
KernelFn kernel_x16_m1(int deg);
KernelFn kernel_x30_m0(int deg);
KernelFn kernel_x30_m1(int deg);
// Latency instances (FP64, one segment, few paths) of R replicas per path:
// size-specialised for n in {3, 4, 5, 6} and {8, 9, 10, 12, 16} (DEG 2 and 3,
// n = 4, 5 also 4), generic for NMAX 8, 16 and 32 (DEG 2, 3, 4 and 6); R = 8 up to
// 8 lanes per replica, 4 up to 16, 2 up to 32.
#define HCX_REP_UNITS(R) \
  KernelFn kernel_rep_xs_r##R(int n, int deg); KernelFn kernel_rep_xl_r##R(int n, int deg); \
  KernelFn kernel_rep_g8_r##R(int deg);
HCX_REP_UNITS(1)
HCX_REP_UNITS(2)
HCX_REP_UNITS(4)
HCX_REP_UNITS(8)
#undef HCX_REP_UNITS
// The same with the evaluation dealt out by columns (DEAL), R = 2 and 4, for
// terms of degree <= 3.
KernelFn kernel_deal_x(int n, int deg, int R);
KernelFn kernel_deal_g(int nmax, int deg, int R);
KernelFn kernel_rep_g16_r1(int deg);
KernelFn kernel_rep_g16_r2(int deg);
KernelFn kernel_rep_g16_r4(int deg);
KernelFn kernel_rep_g32_r1(int deg);
KernelFn kernel_rep_g32_r2(int deg);

}  // namespace hcx
