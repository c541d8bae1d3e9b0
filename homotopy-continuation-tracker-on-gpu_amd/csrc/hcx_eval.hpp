// Evaluation of the path loops: term streams, coefficient staging.
//
// A row's terms are a STREAM per lane: position p of equation i at
// [p][i], all positions of Jacobian column 0, then of column 1, and so on
// (dH/dx), or all terms of the row (dH/dt, H), at their places in the problem's
// tables.  The number of positions is the maximum over the equations; where an
// equation has no term it holds a zero term (a variable index that reads the
// constant 0).  A column begins with the positions up to the last one at which
// some equation has a scalar other than 1 ("scaled"), the rest needs no
// scaling.  Every instance computes a term as ((scalar * coefficient) *
// variable) * variable ... with the roundings of cmul_term and adds the terms
// of a row in stream order, so instances that differ only in where the streams
// live give the same bits.
//
// What bounds it: per term two or three 16-byte LDS gathers and six to ten
// FP64 operations; everything else is overhead, so the records in LDS hold byte offsets
// (no decoding beyond a mask and an add), unscaled positions skip the scaling,
// and the counts come from the kernel arguments.
#pragma once

namespace hcx {
namespace dev {

// The records' byte offsets count 16-byte slots (FP64); FP32 data, in slots of
// 8 bytes, lies at half of them, a shift that the field extraction includes.
template <class T>
constexpr int kHalf = sizeof(T) == 8 ? 0 : 1;
// The value at the low 16 bits (lo) or at bits 16-25 (hi) of a record word.
template <class T>
__device__ __forceinline__ cx<T> lds_lo(const unsigned char* base, uint32_t r) {
  return *reinterpret_cast<const cx<T>*>(base + ((r >> kHalf<T>) & (0xffffu >> kHalf<T>)));
}
template <class T>
__device__ __forceinline__ cx<T> lds_hi(const unsigned char* base, uint32_t r) {
  return *reinterpret_cast<const cx<T>*>(base + ((r >> (16 + kHalf<T>)) & (0x3ffu >> kHalf<T>)));
}

// a * b with the roundings spelled out (they do not depend on what the
// compiler fuses): the products with b.im rounded, those with b.re fused.
__device__ __forceinline__ cx<double> cmul_term(cx<double> a, cx<double> b) {
  return cmk<double>(__builtin_fma(a.re, b.re, -(a.im * b.im)), __builtin_fma(a.im, b.re, a.re * b.im));
}
__device__ __forceinline__ cx<float> cmul_term(cx<float> a, cx<float> b) {
  return cmk<float>(__builtin_fmaf(a.re, b.re, -(a.im * b.im)), __builtin_fmaf(a.im, b.re, a.re * b.im));
}

// Compact records of the throughput instances, in LDS: byte offsets of the
// coefficient slot (16 bits, from the group's coefficient area) and of the
// variables (10 bits, multiples of 16, from its x area), and the scalar s.
//   degree <= 2:  dH/dx  c | v0 << 16 | s << 26
//                 H      c | v0 << 16 | s << 26,  v1 | j << 16
//   degree 3, 4:  dH/dx  c | v0 << 16,  v1 | v2 << 6 | s << 16
//                 H      c | v0 << 16,  v1 | v2 << 16,  v3 | j << 16,  s
//   degree 5, 6:  dH/dx  c | v0 << 16,  v1 | v2 << 16,  v3 | v4 << 16,  s
//                 H      c | v0 << 16 | s << 26,  v1 | v2 << 16 | s' << 26,
//                        v3 | v4 << 16 | s'' << 26,  v5 | j << 16
// with j the coefficient's number (index of dc/dt in global memory); s is of 6
// bits in 26.., of 16 in 16.. and whole in a word of its own; in three parts
// s, s', s'' of 6 bits, the lowest first.
template <int DEG>
struct StreamRec {
  static constexpr int kJ = DEG <= 2 ? 4 : (DEG <= 4 ? 8 : 16);
  static constexpr int kH = DEG <= 2 ? 8 : 16;
  static constexpr int kJWord = DEG <= 2 ? 1 : (DEG <= 4 ? 2 : 3);  // word of j
};
// A record of N bytes.
template <int N>
__device__ __forceinline__ void load_rec(const unsigned char* a, uint32_t (&r)[4]) {
  if constexpr (N == 4) {
    r[0] = *reinterpret_cast<const uint32_t*>(a);
  } else if constexpr (N == 8) {
    const uint2 q = *reinterpret_cast<const uint2*>(a);
    r[0] = q.x;
    r[1] = q.y;
  } else {
    const uint4 q = *reinterpret_cast<const uint4*>(a);
    r[0] = q.x;
    r[1] = q.y;
    r[2] = q.z;
    r[3] = q.w;
  }
}
// The values of a term's NV variables (v0 in the first word's upper half, then
// two per word).
template <int NV, class T>
__device__ __forceinline__ void rec_vars(const unsigned char* xb, const uint32_t (&r)[4], cx<T> (&x)[NV]) {
#pragma unroll
  for (int q = 0; q < NV; ++q) x[q] = q % 2 == 0 ? lds_hi<T>(xb, r[q / 2]) : lds_lo<T>(xb, r[(q + 1) / 2]);
}
// Those of a dH/dx record of the throughput instances.
template <int DEG, class T>
__device__ __forceinline__ void jac_vars(const unsigned char* xb, const uint32_t (&r)[4], cx<T> (&x)[DEG - 1]) {
  if constexpr (DEG <= 2 || DEG > 4) {
    rec_vars<DEG - 1, T>(xb, r, x);
  } else {
    x[0] = lds_hi<T>(xb, r[0]);
    x[1] = *reinterpret_cast<const cx<T>*>(xb + ((r[1] >> kHalf<T>) & (0x3ffu >> kHalf<T>)));
    if constexpr (DEG > 3) x[2] = *reinterpret_cast<const cx<T>*>(xb + (((r[1] >> 10) & 0x3fu) << (4 - kHalf<T>)));
  }
}
template <int DEG>
__device__ __forceinline__ int jac_scalar(const uint32_t (&r)[4]) {
  return DEG <= 2 ? (int)r[0] >> 26 : (DEG <= 4 ? (int)r[1] >> 16 : (int)r[3]);
}
template <int DEG>
__device__ __forceinline__ int h_scalar(const uint32_t (&r)[4]) {
  if constexpr (DEG <= 2) return (int)r[0] >> 26;
  if constexpr (DEG <= 4) return (int)r[3];
  return ((int)r[2] >> 26 << 12) | (int)(r[1] >> 26 << 6) | (int)(r[0] >> 26);
}
// (scalar * coefficient) * variable ..., SC: with a scalar other than 1
template <int NV, bool SC, class T, class S>
__device__ __forceinline__ cx<T> term_value(cx<T> c, S s, const cx<T> (&x)[NV]) {
  if constexpr (SC) c = cscale(c, (T)s);
#pragma unroll
  for (int q = 0; q < NV; ++q) c = cmul_term(c, x[q]);
  return c;
}

// One round over NB columns of a row of dH/dx (throughput instances): term k
// of each, the zero term past a column's last (SC: a scaled position).  All
// records are requested together, then all gathers.  off: byte offset of the
// first column's positions from rp; zero: that of the zero terms.
template <int NMAX, int DEG, bool SC, int JB, int NB, bool PIN, class T>
__device__ __forceinline__ void jac_round(const unsigned char* rp, int n, int off, int zero, const int (&cnt)[NB],
                                          int k, const unsigned char* xb, const unsigned char* cb, cx<T> (&A)[NMAX]) {
  constexpr int RS = StreamRec<DEG>::kJ;
  uint32_t r[NB][4];
  cx<T> c[NB], x[NB][DEG - 1];
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    if (JB + u < NMAX) {
      load_rec<RS>(rp + (k < cnt[u] ? off + k * (n * RS) : zero), r[u]);
      off += cnt[u] * (n * RS);
    }
  }
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    if (JB + u < NMAX) {
      c[u] = lds_lo<T>(cb, r[u][0]);
      jac_vars<DEG, T>(xb, r[u], x[u]);
    }
  }
  // PIN: all gathers before the first product
  if constexpr (PIN) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < NB; ++u)
    if (JB + u < NMAX) A[JB + u] = cadd(A[JB + u], term_value<DEG - 1, SC, T>(c[u], jac_scalar<DEG>(r[u]), x[u]));
}

// Row gl of dH/dx from the compact streams at lt
// (dev-eval-indxing-generalized_3views_4pts.cuh:70-86), NB columns at a time:
// one column after the other, each term is two exposed LDS latencies and each
// column two loops.
template <int NMAX, int DEG, int NB, int JB, bool PIN, class T, class SegT>
__device__ __forceinline__ void eval_jac_blocks(const SegT& S, int n, const unsigned char* rp, int off,
                                                const unsigned char* xb, const unsigned char* cb,
                                                cx<T> (&A)[NMAX]) {
  if constexpr (JB < NMAX) {
    int cnt[NB], end = 0, scaled = 0, tot = 0;
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      cnt[u] = 0;
      if (JB + u < NMAX) {
        const unsigned int cc = S.colc[JB + u];
        cnt[u] = (int)(cc & 0xffffu);
        end = max(end, cnt[u]);
        scaled = max(scaled, (int)(cc >> 16));
        tot += cnt[u];
        A[JB + u] = cmk<T>(0, 0);
      }
    }
    const int zero = S.hx_recs * StreamRec<DEG>::kJ;
    int k = 0;
#pragma unroll 1
    for (; k < scaled; ++k) jac_round<NMAX, DEG, true, JB, NB, PIN, T>(rp, n, off, zero, cnt, k, xb, cb, A);
#pragma unroll 1
    for (; k < end; ++k) jac_round<NMAX, DEG, false, JB, NB, PIN, T>(rp, n, off, zero, cnt, k, xb, cb, A);
    eval_jac_blocks<NMAX, DEG, NB, JB + NB, PIN, T>(S, n, rp, off + tot * (n * StreamRec<DEG>::kJ), xb, cb, A);
  }
}

// Jacobian records of the latency instances: the scalar as the high word of
// its double (the low word is 0), and one row of zero terms after each
// column's positions.
//   degree <= 2:  {c | v0 << 16, s}     degree 3, 4:  {c | v0 << 16, v1 | v2 << 16, s, 0}
//   degree 5, 6:  {c | v0 << 16, v1 | v2 << 16, v3 | v4 << 16, s}
template <int DEG>
struct LatencyRec {
  static constexpr int kJ = DEG <= 2 ? 8 : 16;
  static constexpr int kS = DEG <= 2 ? 1 : (DEG <= 4 ? 2 : 3);  // word of the scalar
};
template <int DEG>
__device__ __forceinline__ double latency_scalar(const uint32_t (&r)[4]) {
  return __longlong_as_double((long long)((unsigned long long)r[LatencyRec<DEG>::kS] << 32));
}

// Row gl of dH/dx on the latency instances (one wave per SIMD: every LDS
// round trip is exposed).  Round by round, one term of every column at once:
// all records of up to eight columns are requested together, then all their
// gathers, so a round costs two LDS latencies instead of two per column.
// Replica s of R takes positions s, s + R, ...; past a column's last position
// it reads the column's zero terms.
template <int NMAX, int DEG, class SegT>
__device__ __forceinline__ void eval_jac_rounds(const SegT& S, int n, int gle, const unsigned char* xb,
                                                const unsigned char* cb, cx<double> (&A)[NMAX],
                                                const unsigned char* lt, int k0, int ks) {
  constexpr int RS = LatencyRec<DEG>::kJ;
  // columns at a time; degree 5 and 6: 5 variables of two columns fill the registers
  constexpr int NB = DEG > 4 ? 2 : (NMAX <= 6 ? NMAX : (NMAX <= 10 ? (NMAX + 1) / 2 : 4));
  const int rounds_end = S.max_terms;
#pragma unroll
  for (int j = 0; j < NMAX; ++j) A[j] = cmk<double>(0, 0);
#pragma unroll 1
  for (int rd = 0; rd < rounds_end; rd += ks) {
    const int k = rd + k0;
    const unsigned char* rp = lt + gle * RS;
#pragma unroll
    for (int jb = 0; jb < NMAX; jb += NB) {
      // generic instances skip the blocks of absent columns (n = 3, degree 5, 1024
      // waves: 6.31 -> 4.59 ms)
      if (DEG > 4 && jb >= n) continue;
      uint32_t r[NB][4];
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        if (jb + u < NMAX) {
          const int cnt = (int)(S.colc[jb + u] & 0xffffu);
          load_rec<RS>(rp + min(k, cnt) * (n * RS), r[u]);
          rp += (cnt + (jb + u < n ? 1 : 0)) * (n * RS);
        }
      }
      cx<double> c[NB], x[NB][DEG - 1];
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        if (jb + u < NMAX) {
          c[u] = lds_lo<double>(cb, r[u][0]);
          rec_vars<DEG - 1, double>(xb, r[u], x[u]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // all gathers before the first product
#pragma unroll
      for (int u = 0; u < NB; ++u)
        if (jb + u < NMAX)
          A[jb + u] = cadd(A[jb + u], term_value<DEG - 1, true, double>(c[u], latency_scalar<DEG>(r[u]), x[u]));
    }
  }
}

// The same with the columns dealt out: replica s of R sums columns s, s + R, ...
// whole (B[i]: column R i + s; past the last column, 0), each in the order of
// its stream, so the sums are those of one replica.  p, end: the lane's place
// in each of its columns and their zero terms.
template <int NMAX, int DEG, int R, int NC, class SegT>
__device__ __forceinline__ void eval_jac_dealt(const SegT& S, int n, int gle, int s, const unsigned char* xb,
                                               const unsigned char* cb, cx<double> (&B)[NC],
                                               const unsigned char* lt) {
  constexpr int RS = LatencyRec<DEG>::kJ;
  constexpr int NB = NC <= 5 ? NC : (NC + 1) / 2;  // columns at a time
  const int rounds_end = S.max_terms, row = n * RS;
  int p[NC], end[NC], off = gle * RS;
  const int none = off + (int)(S.colc[0] & 0xffffu) * row;  // zero terms of column 0
#pragma unroll
  for (int j = 0; j < R * NC; ++j) {
    const int cnt = j < NMAX ? (int)(S.colc[j < NMAX ? j : 0] & 0xffffu) : 0;
    const bool in = j < NMAX && j < n;
    const int b = in ? off : none, z = in ? off + cnt * row : none;
    p[j / R] = (j % R == 0 || s == j % R) ? b : p[j / R];
    end[j / R] = (j % R == 0 || s == j % R) ? z : end[j / R];
    off += in ? (cnt + 1) * row : 0;
  }
#pragma unroll
  for (int i = 0; i < NC; ++i) B[i] = cmk<double>(0, 0);
#pragma unroll 1
  for (int k = 0; k < rounds_end; ++k) {
#pragma unroll
    for (int ib = 0; ib < NC; ib += NB) {
      uint32_t r[NB][4];
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        if (ib + u < NC) {
          load_rec<RS>(lt + p[ib + u], r[u]);
          p[ib + u] = min(p[ib + u] + row, end[ib + u]);
        }
      }
      cx<double> c[NB], x[NB][DEG - 1];
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        if (ib + u < NC) {
          c[u] = lds_lo<double>(cb, r[u][0]);
          rec_vars<DEG - 1, double>(xb, r[u], x[u]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // all gathers before the first product
#pragma unroll
      for (int u = 0; u < NB; ++u)
        if (ib + u < NC)
          B[ib + u] = cadd(B[ib + u], term_value<DEG - 1, true, double>(c[u], latency_scalar<DEG>(r[u]), x[u]));
    }
  }
}

// One chunk of Q terms of a row of dH/dt or H, positions k, k + ks, ...
// (positions past the last read the zero terms that end the stream).  dot:
// this lane's group sums dc/dt (an RK4 stage) instead of c(t): from its LDS
// area at db, or (GDOT) from global memory, requested for the whole chunk
// before the first product.
template <int DEG, bool SC, bool GDOT, int Q, bool PIN, class T>
__device__ __forceinline__ cx<T> rhs_chunk(const unsigned char* rp, int n, int k, int ks, int cnt,
                                                const unsigned char* xb, const unsigned char* cb,
                                                const double2* dg, bool dot, cx<T> acc) {
  constexpr int RS = StreamRec<DEG>::kH;
  uint32_t r[Q][4];
  cx<T> c[Q], x[Q][DEG];
#pragma unroll
  for (int q = 0; q < Q; ++q) load_rec<RS>(rp + min(k + q * ks, cnt) * (n * RS), r[q]);
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    c[q] = lds_lo<T>(cb, r[q][0]);
    rec_vars<DEG, T>(xb, r[q], x[q]);
  }
  if constexpr (GDOT) {
    if (dot) {
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const double2 d = dg[r[q][StreamRec<DEG>::kJWord] >> 16];
        c[q] = cmk<T>((T)d.x, (T)d.y);
      }
    }
  }
  // PIN: every load of the chunk is requested before the first product, also
  // where the compiler would rather save registers
  if constexpr (PIN) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int q = 0; q < Q; ++q) acc = cadd(acc, term_value<DEG, SC, T>(c[q], h_scalar<DEG>(r[q]), x[q]));
  return acc;
}

// Row gl of sum_k s * coef * prod x over the dH/dt streams (…cuh:89-120):
// H with c(t), dH/dt with dc/dt.
template <int DEG, bool GDOT, int Q, bool PIN, class T, class SegT>
__device__ __forceinline__ cx<T> eval_rhs_stream(const SegT& S, int n, int gle, const unsigned char* xb,
                                                      const unsigned char* cb, const unsigned char* db,
                                                      const double2* dg, bool dot, const unsigned char* lt, int k0,
                                                      int ks) {
  const unsigned char* base = (!GDOT && dot) ? db : cb;
  const unsigned char* rp = lt + S.tab_h + gle * StreamRec<DEG>::kH;
  const int cnt = S.htT;
  cx<T> acc = cmk<T>(0, 0);
  int k = 0;
#pragma unroll 1
  for (; k < S.htS; k += Q * ks) acc = rhs_chunk<DEG, true, GDOT, Q, PIN, T>(rp, n, k + k0, ks, cnt, xb, base, dg, dot, acc);
#pragma unroll 1
  for (; k < cnt; k += Q * ks) acc = rhs_chunk<DEG, false, GDOT, Q, PIN, T>(rp, n, k + k0, ks, cnt, xb, base, dg, dot, acc);
  return acc;
}

// sum over positions k0, k0 + ks, ... < cnt of a stream of full Term records
// (n apart from tp; global memory or an LDS copy).  The records of a chunk
// are requested before the first is used.  CLAMP (records in global memory):
// past the last position that position again, not added, so a chunk has no
// branches; from LDS, where a record costs little, the branches are cheaper than
// the products.  GDOT: lanes with dot take dc/dt
// from global memory (dg, indexed by the coefficient numbers ci).
template <int NV, bool GDOT, bool CLAMP, class T>
__device__ __forceinline__ cx<T> term_stream_sum(const Term* tp, int cnt, int n, const cx<T>* sx,
                                                      const cx<T>* coef, const double2* dg, const int* ci,
                                                      bool dot, int k0, int ks) {
  cx<T> acc = cmk<T>(0, 0);
  for (int kb = k0; kb < cnt; kb += kTermChunk * ks) {
    Term tm[kTermChunk];
    int cj[kTermChunk];
    cx<T> c[kTermChunk];
#pragma unroll
    for (int q = 0; q < kTermChunk; ++q) {
      const int k = kb + q * ks;
      const size_t at = (size_t)(CLAMP ? min(k, cnt - 1) : k) * n;
      if (CLAMP || k < cnt) {
        tm[q] = tp[at];
        if constexpr (GDOT) cj[q] = ci[at];
      }
    }
#pragma unroll
    for (int q = 0; q < kTermChunk; ++q)
      if (CLAMP || kb + q * ks < cnt) c[q] = coef[tm[q].c];
    if constexpr (GDOT) {
      if (dot) {
#pragma unroll
        for (int q = 0; q < kTermChunk; ++q)
          if (CLAMP || kb + q * ks < cnt) {
            const double2 d = dg[cj[q]];
            c[q] = cmk<T>((T)d.x, (T)d.y);
          }
      }
    }
#pragma unroll
    for (int q = 0; q < kTermChunk; ++q) {
      if (!CLAMP && kb + q * ks >= cnt) continue;
      cx<T> v = cscale(c[q], (T)tm[q].s);
#pragma unroll
      for (int d = 0; d < NV; ++d) v = cmul_term(v, sx[term_var(tm[q], d)]);
      const cx<T> sum = cadd(acc, v);
      if (kb + q * ks < cnt) acc = sum;
    }
  }
  return acc;
}

// Row gl of dH/dx from the full records: those of the LDS copy at tl, or in
// global memory (tl null).
template <int NMAX, int DEG, class T, class SegT>
__device__ __forceinline__ void eval_jac_terms(const SegT& S, int n, int gle, const cx<T>* sx,
                                               const cx<T>* sc, cx<T> (&A)[NMAX], const Term* tl, int k0,
                                               int ks) {
  size_t off = gle;
#pragma unroll
  for (int j = 0; j < NMAX; ++j) {
    cx<T> acc = cmk<T>(0, 0);
    if (j < n) {
      int cnt;
      if (S.hx_cnt) {
        cnt = S.hx_cnt[j];
      } else {
        cnt = (int)(S.colc[j] & 0xffffu);
      }
      if (tl)
        acc = term_stream_sum<DEG - 1, false, false, T>(tl + off, cnt, n, sx, sc, nullptr, nullptr, false, k0, ks);
      else
        acc = term_stream_sum<DEG - 1, false, true, T>(S.hx + off, cnt, n, sx, sc, nullptr, nullptr, false, k0, ks);
      off += (size_t)cnt * n;
    }
    A[j] = acc;
  }
}

// Row gl of dH/dt or H from the full records (base: c(t) or dc/dt in LDS).
template <int DEG, bool GDOT, class T, class SegT>
__device__ __forceinline__ cx<T> eval_rhs_terms(const SegT& S, int n, int gle, const cx<T>* sx,
                                                     const cx<T>* base, const double2* dg, bool dot,
                                                     const Term* tl, int k0, int ks) {
  const int* ci = S.ht_ci + gle;
  if (tl) return term_stream_sum<DEG, GDOT, false, T>(tl + (size_t)S.hx_recs + gle, S.htT, n, sx, base, dg, ci, dot, k0, ks);
  return term_stream_sum<DEG, GDOT, true, T>(S.ht + gle, S.htT, n, sx, base, dg, ci, dot, k0, ks);
}

// ------------------------------------------------------------ staging
// LDS byte offset of coefficient j from the group's region.  A coefficient
// that no term uses has no slot: it goes to offset 0, x's first slot, which
// is published after the staging (no branch per coefficient).  SL: the list is
// in LDS with the compact tables; head: offset of the coefficient area.
template <bool SL, class SegT>
__device__ __forceinline__ uint32_t slot_offset(const SegT& S, const unsigned char* lt, int j, int head) {
  if constexpr (SL) {
    return reinterpret_cast<const unsigned short*>(lt + S.tab_slot)[j];
  } else {
    const int q = S.cslot[j];
    return q < S.nslot ? (uint32_t)(head + q * 16) : 0u;
  }
}

// c_j(t) of order MC in t and (dot) dc_j/dt(t) into the group's LDS slots, Q of
// the lane's coefficients at a time: all of a chunk's loads are requested
// before the first is used, so the staging costs one memory latency per Q
// coefficients; full chunks address with constant offsets, the last
// coefficients go as one chunk.  hx, ht: the instance's tables; xb: where the
// offsets of T's slots count from, db: from a slot of c to that of dc/dt.
template <int MC, int Q, bool SL, class T, class SegT>
__device__ __forceinline__ void stage_chunks(const SegT& S, const Group& g, const double2* hx, const double2* ht,
                                             double t, unsigned char* xb, int head, int db, bool dot,
                                             const unsigned char* lt) {
  const int C1 = S.C + 1, st = g.G * g.R;
  auto put = [&](const double2* a, uint32_t o) {
    double cr = a[MC].x, ci = a[MC].y;
#pragma unroll
    for (int m = MC - 1; m >= 0; --m) {
      cr = cr * t + a[m].x;
      ci = ci * t + a[m].y;
    }
    *reinterpret_cast<cx<T>*>(xb + (o >> kHalf<T>)) = cmk<T>((T)cr, (T)ci);
  };
  auto put_dot = [&](const double2* b, uint32_t o) {
    double dr = b[MC - 1].x, di = b[MC - 1].y;
#pragma unroll
    for (int m = MC - 2; m >= 0; --m) {
      dr = dr * t + b[m].x;
      di = di * t + b[m].y;
    }
    if (o) *reinterpret_cast<cx<T>*>(xb + db + (o >> kHalf<T>)) = cmk<T>((T)dr, (T)di);
  };
  int j = g.gl + g.s * g.G;
  const double2* ha = hx + (size_t)j * (MC + 1);
  const double2* hb = ht + (size_t)j * MC;
#pragma unroll 1
  for (; j + (Q - 1) * st < C1; j += Q * st) {
    double2 a[Q][MC + 1], b[Q][MC];
    uint32_t o[Q];
#pragma unroll
    for (int u = 0; u < Q; ++u) {
#pragma unroll
      for (int m = 0; m <= MC; ++m) a[u][m] = ha[u * st * (MC + 1) + m];
      o[u] = slot_offset<SL>(S, lt, j + u * st, head);
    }
    if (dot) {
#pragma unroll
      for (int u = 0; u < Q; ++u)
#pragma unroll
        for (int m = 0; m < MC; ++m) b[u][m] = hb[u * st * MC + m];
    }
#pragma unroll
    for (int u = 0; u < Q; ++u) put(a[u], o[u]);
    if (dot) {
#pragma unroll
      for (int u = 0; u < Q; ++u) put_dot(b[u], o[u]);
    }
    ha += Q * st * (MC + 1);
    hb += Q * st * MC;
  }
  // the rest, fewer than Q: as one chunk whose surplus repeats the last
  // coefficient
  if (j < C1) {
    constexpr int Q1 = Q > 1 ? Q - 1 : 1;
    double2 a[Q1][MC + 1], b[Q1][MC];
    uint32_t o[Q1];
#pragma unroll
    for (int u = 0; u < Q1; ++u) {
      const int d = j + u * st < C1 ? u * st : 0;
#pragma unroll
      for (int m = 0; m <= MC; ++m) a[u][m] = ha[d * (MC + 1) + m];
      o[u] = slot_offset<SL>(S, lt, j + d, head);
      if (dot) {
#pragma unroll
        for (int m = 0; m < MC; ++m) b[u][m] = hb[d * MC + m];
      }
    }
#pragma unroll
    for (int u = 0; u < Q1; ++u) put(a[u], o[u]);
    if (dot) {
#pragma unroll
      for (int u = 0; u < Q1; ++u) put_dot(b[u], o[u]);
    }
  }
}

// Coefficient polynomials in t of the group's instance into LDS
// (eval_parameter_homotopy, …cuh:34-67).  Coefficient j goes to slot
// cslot[j]: slots follow the order in which the rows of a group read them
// (term by term), so the lanes of a group that read term k of their rows
// together hit consecutive LDS words instead of words one equation apart.  The
// replicas of a group share its LDS region and stage every R-th coefficient
// each.  Q: coefficients in flight per lane at order 1 (fewer at higher
// orders, by their registers).  Computed in FP64 and stored as T: at FP64 the
// offsets count from the group's region, at FP32 (half of them) from the middle of
// what precedes the coefficient area, so that the area begins at the same place
// and an unused coefficient goes to x's slots past those that FP32 uses.
template <bool SL, int Q, class T, class SegT>
__device__ __forceinline__ void stage_coeffs(const SegT& S, const Group& g, const double2* hx, const double2* ht,
                                               double t, unsigned char* xb, int head, int db, bool dot,
                                               const unsigned char* lt) {
  constexpr int Q2 = Q > 2 ? Q / 2 : 1, Q3 = Q > 3 ? Q / 3 : 1;
  switch (S.M) {
    case 1: return stage_chunks<1, Q, SL, T>(S, g, hx, ht, t, xb, head, db, dot, lt);
    case 2: return stage_chunks<2, Q2, SL, T>(S, g, hx, ht, t, xb, head, db, dot, lt);
    case 3: return stage_chunks<3, Q3, SL, T>(S, g, hx, ht, t, xb, head, db, dot, lt);
    case 4: return stage_chunks<4, Q3, SL, T>(S, g, hx, ht, t, xb, head, db, dot, lt);
    default: break;
  }
  const int C1 = S.C + 1, M = S.M;
  for (int j = g.gl + g.s * g.G; j < C1; j += g.G * g.R) {
    const uint32_t o = slot_offset<SL>(S, lt, j, head);
    const double2* ha = hx + (size_t)j * (M + 1);
    double cr = ha[M].x, ci = ha[M].y;
    for (int m = M - 1; m >= 0; --m) {
      cr = cr * t + ha[m].x;
      ci = ci * t + ha[m].y;
    }
    *reinterpret_cast<cx<T>*>(xb + (o >> kHalf<T>)) = cmk<T>((T)cr, (T)ci);
    if (dot && o) {
      const double2* hb = ht + (size_t)j * M;
      double dr = hb[M - 1].x, di = hb[M - 1].y;
      for (int m = M - 2; m >= 0; --m) {
        dr = dr * t + hb[m].x;
        di = di * t + hb[m].y;
      }
      *reinterpret_cast<cx<T>*>(xb + db + (o >> kHalf<T>)) = cmk<T>((T)dr, (T)di);
    }
  }
}

// x and the constants 1 and 0 (variable indices n and n + 1).
template <class T>
__device__ __forceinline__ void publish_x(cx<T>* sx, cx<double> x, const Group& g, int n, bool act, bool row) {
  if (act && row) sx[g.gl] = ccast<T>(x);
  if (act && g.gl == 0) {
    sx[n] = cmk<T>(T(1), T(0));
    sx[n + 1] = cmk<T>(T(0), T(0));
  }
}

}  // namespace dev
}  // namespace hcx
