// Kernels and per-precision launchers of the axhelm operator, shared by the
// translation units that instantiate them (nbx_axhelm.hip: FP64,
// nbx_axhelm_f32.hip: FP32, nbx_axhelm_bf16.hip: bf16 geometry), so that the
// instantiations for N = 1..15 compile in parallel.  See nbx_axhelm.hip for
// the operator, its mapping and its arithmetic order.
#pragma once
#include "nbx_internal.h"
#include "nbx_reduce.h"
#include <cstring>
#include <cstdio>
#include <type_traits>
#include <cstdlib>

namespace nbx {

template <typename T>
__device__ __forceinline__ T fmaT(T a, T b, T c);
template <>
__device__ __forceinline__ double fmaT<double>(double a, double b, double c) { return __builtin_fma(a, b, c); }
template <>
__device__ __forceinline__ float fmaT<float>(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// Load of a geometric factor / lambda stored as G, converted to the math type T.
// bf16 is stored as its 16 high bits (uint16_t).
template <typename T, typename G>
__device__ __forceinline__ T ldg(const G* p);
template <>
__device__ __forceinline__ double ldg<double, double>(const double* p) { return ldnt(p); }
template <>
__device__ __forceinline__ float ldg<float, float>(const float* p) { return ldnt(p); }
template <>
__device__ __forceinline__ float ldg<float, uint16_t>(const uint16_t* p)
{
  return __uint_as_float((uint32_t)ldnt(p) << 16);
}
// NT = false: an ordinary (cached) load, for data that other lanes of the
// workgroup read again right away
template <typename T, typename G, bool NT>
__device__ __forceinline__ T ldgc(const G* p)
{
  if constexpr (NT) {
    return ldg<T, G>(p);
  } else if constexpr (sizeof(G) == 2) {
    return __uint_as_float((uint32_t)(*p) << 16);
  } else {
    return (T)(*p);
  }
}

// LDS places of node (i, j, k).  r array: i + j RS + k PS with RS odd, so a
// lane per r line (address t RS) meets no bank conflict; s array: i + j NQ + k
// QS with QS = NQ modulo the slots one LDS cycle serves (128 bytes), so lanes
// over nodes and lanes over s lines both read consecutive slots.
template <typename T, int NQ>
struct LineLayout {
  static constexpr int RS = NQ | 1, PS = NQ * RS, SZ = NQ * PS;
  static constexpr int M = 128 / (int)sizeof(T);
  static constexpr int QS = NQ * NQ + ((NQ - NQ * NQ) % M + M) % M, SS = NQ * QS;
};

// Row i of D through the constant address space: uniform addresses become
// scalar loads and the row's values scalar operands of the products.  The
// pointer is made opaque at every row, or the compiler keeps all of D in
// scalar registers from the first use to the last and spills them.
template <typename T>
using ConstPtr = const T __attribute__((address_space(4)))*;
template <typename T, int NQ>
struct DRow {
  T d[NQ];
  __device__ __forceinline__ void load(ConstPtr<T> D, int row)
  {
    asm volatile("" : "+s"(D));
#pragma unroll
    for (int m = 0; m < NQ; ++m) d[m] = D[row * NQ + m];
  }
};

// The geometric factors and lambda0 of the lane's column, one slab at a time,
// fetched AHEAD slabs before their use.  NT: nontemporal loads (single use);
// cached ones where other workgroups of the XCD read the same element.
template <typename T, int NQ, bool BK, typename G, bool NT, int AHEAD, typename IDX>
struct GeoStream {
  static constexpr int NQ2 = NQ * NQ, NP = NQ2 * NQ;
  const G *g, *l0, *l1;  // element bases (uniform in the workgroup)
  IDX go, lo;            // the lane's node (k = 0) past them
  T Gk[AHEAD][7];
  __device__ __forceinline__ void fetch(int k)
  {
    const int n = k * NQ2;
    T(&u)[7] = Gk[k % AHEAD];
    u[0] = ldgc<T, G, NT>(&(g + kG00 * NP)[go + n]);
    u[1] = ldgc<T, G, NT>(&(g + kG01 * NP)[go + n]);
    u[2] = ldgc<T, G, NT>(&(g + kG02 * NP)[go + n]);
    u[3] = ldgc<T, G, NT>(&(g + kG11 * NP)[go + n]);
    u[4] = ldgc<T, G, NT>(&(g + kG12 * NP)[go + n]);
    u[5] = ldgc<T, G, NT>(&(g + kG22 * NP)[go + n]);
    if (!BK) u[6] = ldgc<T, G, NT>(&l0[lo + n]);
  }
  __device__ __forceinline__ void begin()
  {
#pragma unroll
    for (int k = 0; k < AHEAD && k < NQ; ++k) fetch(k);
  }
  __device__ __forceinline__ void next(int k)
  {
    if (k + AHEAD < NQ) fetch(k + AHEAD);
  }
  __device__ __forceinline__ T f(int k, int c) const { return Gk[k % AHEAD][c]; }
  __device__ __forceinline__ T lam(int k) const { return Gk[k % AHEAD][6]; }
  __device__ __forceinline__ T mass(int k) const
  {
    const int n = k * NQ2;
    return ldgc<T, G, NT>(&(g + kGWJ * NP)[go + n]) * ldgc<T, G, NT>(&l1[lo + n]);
  }
};

// The same for three fields of one element, read once: the factors of every
// slab stay in registers, lambda0 and GWJ lambda1 in LDS (each lane its own
// column, so without a barrier).
template <typename T, int NQ, bool BK, typename G, typename IDX>
struct GeoKept {
  static constexpr int NQ2 = NQ * NQ;
  GeoStream<T, NQ, true, G, true, NQ, IDX> s;
  T *l, *w;
  __device__ __forceinline__ void load()
  {
    s.begin();
    if constexpr (!BK) {
#pragma unroll
      for (int k = 0; k < NQ; ++k) {
        l[k * NQ2] = ldg<T, G>(&s.l0[s.lo + k * NQ2]);
        w[k * NQ2] = s.mass(k);
      }
    }
  }
  __device__ __forceinline__ void begin() {}
  __device__ __forceinline__ void next(int) {}
  __device__ __forceinline__ T f(int k, int c) const { return s.Gk[k][c]; }
  __device__ __forceinline__ T lam(int k) const { return l[k * NQ2]; }
  __device__ __forceinline__ T mass(int k) const { return w[k * NQ2]; }
};

// One field of one element in line form: a lane is the owner of a node column
// (i, j) = (t % NQ, t / NQ), of an r line and of an s line in turn.  A
// contraction reads its line once, forms all NQ outputs with D's rows as
// scalar operands and writes them back in place, so every node moves through
// LDS 15 times in all; with a lane per output, each derivative read NQ values
// (4 NQ reads a node, and D), and from N = 4 up LDS and registers, not HBM,
// were the bound.  12e6 nodes, one field, before -> now: FP64 BK N = 5
// 335 -> 138 us, N = 7 142 -> 125, N = 12 208 -> 155, N = 15 303 -> 155;
// non-BK N = 12 626 -> 204; FP32 non-BK N = 6 154 -> 101; three fields FP64
// non-BK N = 7 501 -> 266, N = 9 723 -> 377, N = 12 1884 -> 389.  One field
// moves 5.0 to 6.0 TB/s now, HBM-bound.  Each output is the fma chain over m
// (or k) in increasing order, as the oracle has it.
// rq: q of the lane's column on entry; after_forward() may replace it (the
// next field's); q_again(mq) gives q once more for the mass term, before the
// transposed contractions or, with LATE, after them.  EARLY: the first slabs of
// factors are fetched before the forward contractions (AxShape::early).
template <typename T, int NQ, bool BK, bool LATE = false, bool EARLY = false, typename GEO, typename F1, typename F2>
__device__ __forceinline__ void axhelm_lines(const int t, T (&rq)[NQ], T (&out)[NQ], ConstPtr<T> D, T* s_r, T* s_s,
                                             GEO& geo, F1&& after_forward, F2&& q_again)
{
  using LL = LineLayout<T, NQ>;
  constexpr int RS = LL::RS, PS = LL::PS, QS = LL::QS;
  const int a = t % NQ, b = t / NQ;
  T* const nr = s_r + b * RS + a;  // node (a, b, k) at + k PS
  T* const ns = s_s + t;           // the same node, at + k QS
  T* const lr = s_r + t * RS;      // r line (j, k) = (a, b)
  T* const ls = s_s + b * QS + a;  // s line (i, k) = (a, b), node j at + j NQ
  const T* const lq = s_r + b * PS + a;  // the same line of q
  T v[NQ];
  {
    T ql[NQ], qm[NQ];
#pragma unroll
    for (int k = 0; k < NQ; ++k) nr[k * PS] = rq[k];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < NQ; ++m) {
      ql[m] = lr[m];
      qm[m] = lq[m * RS];
    }
    __syncthreads();
    if (EARLY) geo.begin();
    DRow<T, NQ> R, Rn;
    R.load(D, 0);
    T qr, qs;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      // the first products wait for row i; then the previous row's results
      // and the next row's loads are issued, in flight during the rest
      T pr = qr, ps = qs;
      qr = fmaT(R.d[0], ql[0], T(0));
      qs = fmaT(R.d[0], qm[0], T(0));
      T qt = fmaT(R.d[0], rq[0], T(0));
      __builtin_amdgcn_sched_barrier(0);
      if (i > 0) {
        lr[i - 1] = pr;
        ls[(i - 1) * NQ] = ps;
      }
      if (i + 1 < NQ) Rn.load(D, i + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 1; m < NQ; ++m) {
        qr = fmaT(R.d[m], ql[m], qr);
        qs = fmaT(R.d[m], qm[m], qs);
        qt = fmaT(R.d[m], rq[m], qt);
      }
      v[i] = qt;
      R = Rn;
    }
    lr[NQ - 1] = qr;
    ls[(NQ - 1) * NQ] = qs;
  }
#pragma unroll
  for (int k = 0; k < NQ; ++k) out[k] = T(0);
  after_forward();
  __syncthreads();
  {
    if (!EARLY) geo.begin();
    DRow<T, NQ> R, Rn;
    R.load(D, 0);
    T qr = nr[0], qs = ns[0], qrn, qsn;
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const T G01 = geo.f(k, 1), G02 = geo.f(k, 2), G12 = geo.f(k, 4), qt = v[k];
      T Gr = fmaT(G02, qt, fmaT(G01, qs, geo.f(k, 0) * qr));
      T Gs = fmaT(G12, qt, fmaT(geo.f(k, 3), qs, G01 * qr));
      T Gt = fmaT(geo.f(k, 5), qt, fmaT(G12, qs, G02 * qr));
      if (!BK) {
        const T lam0 = geo.lam(k);
        Gr = lam0 * Gr;
        Gs = lam0 * Gs;
        Gt = lam0 * Gt;
      }
      out[0] = fmaT(R.d[0], Gt, out[0]);
      __builtin_amdgcn_sched_barrier(0);
      nr[k * PS] = Gr;
      ns[k * QS] = Gs;
      if (k + 1 < NQ) {
        Rn.load(D, k + 1);
        qrn = nr[(k + 1) * PS];
        qsn = ns[(k + 1) * QS];
      }
      geo.next(k);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 1; m < NQ; ++m) out[m] = fmaT(R.d[m], Gt, out[m]);
      R = Rn;
      qr = qrn;
      qs = qsn;
    }
  }
  __syncthreads();
  T mq[NQ];
  if (!LATE) q_again(mq);
  {
    T ar[NQ], as[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) ar[i] = as[i] = T(0);
    DRow<T, NQ> R, Rn;
    R.load(D, 0);
    T gr = lr[0], gs = ls[0], grn, gsn;
#pragma unroll
    for (int m = 0; m < NQ; ++m) {
      ar[0] = fmaT(R.d[0], gr, ar[0]);
      as[0] = fmaT(R.d[0], gs, as[0]);
      __builtin_amdgcn_sched_barrier(0);
      if (m + 1 < NQ) {
        Rn.load(D, m + 1);
        grn = lr[m + 1];
        gsn = ls[(m + 1) * NQ];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 1; i < NQ; ++i) {
        ar[i] = fmaT(R.d[i], gr, ar[i]);
        as[i] = fmaT(R.d[i], gs, as[i]);
      }
      // the step's sums are opaque here: otherwise nothing holds the products
      // to their step, they move behind the last row's loads, and every row of
      // D spills (126 scalar registers in vector lanes for FP64 Helmholtz at
      // N = 9, 464 at N = 15; 0 and 16 now; N = 9, 1e6 nodes: 18.2 -> 17.4 us)
#pragma unroll
      for (int i = 0; i < NQ; ++i) asm volatile("" : "+v"(ar[i]), "+v"(as[i]));
      R = Rn;
      gr = grn;
      gs = gsn;
    }
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      lr[i] = ar[i];
      ls[i * NQ] = as[i];
    }
  }
  __syncthreads();
  if (LATE) q_again(mq);
#pragma unroll
  for (int k = 0; k < NQ; ++k) {
    T res = (nr[k * PS] + ns[k * QS]) + out[k];
    if (!BK) {
      res = fmaT(geo.mass(k), mq[k], res);
    }
    out[k] = res;
  }
}


// ---- launch shapes ---------------------------------------------------------
// Elements per workgroup (threadIdx.y = slot): enough to fill two to four
// waves with few idle lanes, no more (a workgroup's waves wait for each other
// at five barriers; N = 1 with 64 instead of 32 elements cost 8 % at 37500).
// ahead: slabs of factors in flight, four; two where FP64 would drop below
// three waves per SIMD; all eight at N = 7 FP64 Poisson (177 against 179 us for
// 32768 elements); six at N = 10 FP64 Helmholtz (one field, 2e6 nodes: 33.0
// against 35 us with four); eight at N = 11 with bf16 geometry, Helmholtz
// (1e6 nodes 13.4 -> 11.6 us, 8e6 49.7 -> 47.0; Poisson gains at 1e6 only and
// loses 6 to 13 % from 8e6 on).
// early: the first slabs are fetched before the forward contractions, so that
// memory works during them, and q through the caches (a solver has just
// written it).  One field, us, fetched after them with nontemporal q / now
// (the column form that preceded the line form in brackets), 8e6 nodes:
//   FP64 Poisson    N = 7  81.6 / 77.0 (84.0)    N = 9  91.2 / 83.0 (99.8)
//                   N = 10 97.1 / 86.1 (94.5)
//   FP64 Helmholtz  N = 9  127.4 / 116.2 (123.6) N = 10 130.1 / 119.5 (119.3)
//   FP32 Poisson    N = 7  41.1 / 40.1 (41.8), 17e6 87.3 / 82.3 (84.2)
//                   N = 10 49.6 / 45.1 (47.9)
//   FP32 Helmholtz  N = 10 68.1 / 63.7 (65.0)
// N = 11 and 13 FP64 lose 3 to 6 % by it (their registers leave two waves),
// and bf16 geometry has fewer bytes to wait for (0 to 17 % slower).
// Slower than the column form are only FP64 Helmholtz at N = 10 on half of
// 8e6 nodes by a list (63.7 against 62.0 us), and on 17e6 nodes in buffers that
// no cache holds (266 against 262), and bf16 Poisson at N = 11 on 1e6 nodes
// (12.2 against 12.0).
template <typename T, int NQ, bool BK, typename G = T>
struct AxShape {
  static constexpr bool f64 = sizeof(T) == 8;
  static constexpr int epb = NQ == 2 ? 32 : NQ == 3 ? 14 : NQ == 4 ? 8 : NQ == 5 ? 5 : NQ == 6 ? 3 : 1;
  static constexpr int ahead = f64 && (NQ >= 12 || (NQ == 9 && !BK))       ? 2
                               : f64 && NQ == 11 && !BK                    ? 6
                               : (f64 && NQ == 8 && BK)                    ? 8
                               : (sizeof(G) == 2 && NQ == 12 && !BK)       ? 8
                                                                           : 4;
  static constexpr bool early = sizeof(G) != 2 && NQ <= 11;
};
// Three fields: the element's factors kept in registers for all of them
// (k_axhelm_kept) against one workgroup per field (k_axhelm), whose second
// and third read of the factors come from L2 at about 9 TB/s at most.  Three
// times the workgroups are better while the chip is not full.  us, kept / per
// field:
//                       3e5 nodes     1e6           3e6           12e6
//   FP64 Poisson  N = 1 7.2 / 7.1     24.8 / 21.0   69.2 / 60.2   264 / 283
//                 N = 3 8.0 / 6.6     16.9 / 18.6   46.7 / 48.0   165 / 219
//                 N = 5 10.1 / 8.0    22.5 / 22.1   55.6 / 58.6   183 / 259
//                 N = 7 9.9 / 7.6     19.1 / 20.5   56.1 / 51.3   178 / 219
//                 N = 9 16.3 / 9.9    24.8 / 25.1   65.9 / 64.3   216 / 271
//        Helmholtz N = 5 11.3 / 9.6   32.1 / 26.2   76.6 / 72.8   275 / 337
//                 N = 7 11.3 / 9.1    23.1 / 24.5   63.9 / 65.0   231 / 298
//                 N = 8 16.3 / 12.5   38.7 / 33.1   89.5 / 91.7   318 / 419
//   FP32 Poisson  N = 2 6.8 / 7.2     16.3 / 19.1   45.2 / 51.1   166 / 211
//                 N = 7 7.9 / 5.0     11.7 / 9.4    30.2 / 26.0   93 / 101
//        Helmholtz N = 4 8.1 / 6.2    17.1 / 16.1   46.4 / 43.8   162 / 203
// The lines are in waves of elements' lanes (Nq^2 an element, eight waves a
// SIMD are 8192).  The FP64 non-BK form at N = 9 would spill and is per field,
// the FP32 form at N = 1 is slower throughout (198 / 156 at 12e6).
template <typename T, int NQ, bool BK>
struct AxKept {
  static constexpr bool f64 = sizeof(T) == 8;
  static constexpr bool value = f64 ? NQ <= 9 || (NQ == 10 && BK) : NQ <= 8;  // (the PCG form too)
  static constexpr int epb = NQ == 2 ? 32 : NQ == 3 ? 14 : NQ == 4 ? 8 : NQ == 5 ? 5 : NQ == 6 ? 3 : 1;
  static constexpr int waves = f64 && NQ >= 7 ? 2 : 1;
  static constexpr int64_t from =
      f64 ? (NQ == 2 ? 32768 : NQ == 3 ? 16384 : NQ == 5 || NQ == 6 ? 8192 : NQ == 9 ? 6144 : 1536)
          : (NQ == 2 ? INT64_MAX / 64 : NQ == 3 ? 1024 : 8192);
  static bool when(int64_t Nelements) { return Nelements * (NQ * NQ) >= 64 * from; }
};

// Three-field PCG form: one thread group per field of an element against the
// fields in turn.  Groups are faster while the chip is not full, and where the
// fields in turn leave one wave per SIMD.  us, groups / in turn:
//                            1e5 nodes     1e6           3e6           8e6
//   FP64 Poisson   N = 5     6.7 / 9.8     30.0 / 33.2   82.6 / 81.4   236 / 198
//                  N = 7     7.2 / 10.3    29.3 / 27.4   72.7 / 74.4   210 / 179
//                  N = 8     8.8 / 13.0    32.0 / 44.2   80.1 / 102    240 / 245
//                  N = 9     10.6 / 14.3   44.1 / 34.6   120 / 94.3    341 / 225
//                  N = 10    12.2 / 16.6   42.5 / 43.5   114 / 118     330 / 299
//                  N = 11    13.5 / 19.0   47.0 / 57.2   106 / 125     320 / 325
//                  N = 13    21.5 / 26.9   50.9 / 67.5   125 / 167     345 / 414
//        Helmholtz N = 7     7.2 / 10.5    32.2 / 31.3   97.5 / 84.6   262 / 204
//                  N = 8     9.2 / 13.9    35.2 / 48.7   109 / 115     293 / 275
//   FP32 Poisson   N = 7     5.9 / 8.7     22.7 / 22.4   58.1 / 58.7   157 / 143
//                  N = 9     8.7 / 13.0    26.2 / 31.1   69.1 / 90.3   186 / 223
//   bf16 geometry  N = 4     6.7 / 8.7     32.1 / 29.2   86.4 / 78.1   240 / 195  (Helmholtz)
//                  N = 5     5.9 / 9.2     24.0 / 26.2   60.1 / 68.1   151 / 165  (Poisson)
//                  N = 9     9.5 / 15.6    38.5 / 32.6   94.6 / 85.3   271 / 214  (Helmholtz)
//                  N = 9     9.1 / 14.7    27.1 / 30.7   72.5 / 80.8   197 / 193  (Poisson)
//                  N = 13    16.9 / 25.3   42.8 / 43.3   111 / 94.4    279 / 228  (Poisson)
// Each line (in waves of Nq^2 lanes an element) lies between the measured sizes
// on its two sides; kAll: groups at every size, the fields in turn are not built.
template <typename T, int NQ, bool BK, typename G>
struct AxFieldGroups {
  static constexpr bool fits = NQ >= 4 && 3 * (LineLayout<T, NQ>::SZ + LineLayout<T, NQ>::SS) * sizeof(T) < 150000;
  static constexpr int64_t kAll = INT64_MAX / 64;
  static constexpr int64_t below = sizeof(T) == 8   ? (NQ >= 12 ? kAll : NQ == 9 || NQ == 11 ? 8192 : NQ == 6 ? 4096 : 768)
                                   : sizeof(G) == 4 ? (NQ >= 9 ? kAll : 12288)
                                   : NQ == 5 || NQ == 7 || NQ == 8 ? 1024
                                   : NQ == 10                      ? (BK ? 8192 : 1024)
                                   : NQ == 11                      ? 2048
                                   : NQ == 14 && BK                ? 2048
                                   : NQ == 15                      ? 8192
                                                                   : kAll;
  static constexpr bool always = fits && below == kAll;
  static bool when(int64_t Nelements) { return always || Nelements * (NQ * NQ) < 64 * below; }
};

// The elements of a workgroup: a uniform base and a lane offset, so that the
// loads take a scalar base and one 32-bit lane register; with an element list
// and several slots the offset is 64 bits wide.  An idle slot of the last
// workgroup works on its last element and stores nothing (every lane reaches
// the barriers).
template <bool PARTIAL, int EPB>
struct ElemPlace {
  using IDX = typename std::conditional<PARTIAL && (EPB > 1), int64_t, int32_t>::type;
  int64_t base;
  IDX rel;
  bool active;
  __device__ __forceinline__ ElemPlace(int32_t first, int32_t Nelements, const int32_t* elementList, int slot)
  {
    const int32_t s = EPB == 1 ? 0 : min(slot, Nelements - 1 - first);
    active = EPB == 1 || s == slot;
    if constexpr (PARTIAL && EPB > 1) {
      base = 0;
      rel = elementList[first + s];
    } else if constexpr (PARTIAL) {
      base = elementList[first];
      rel = 0;
    } else {
      base = first;
      rel = s;
    }
  }
};

// Aq = A q, one field per workgroup.  Three fields: workgroups of one element
// follow each other on one XCD (workgroup b runs on XCD b % 8), so its L2
// serves the factors to the second and third.
template <typename T, int NQ, int NF, bool BK, bool PARTIAL, typename G>
__global__ __launch_bounds__((NQ * NQ * AxShape<T, NQ, BK>::epb)) void k_axhelm(
    const int32_t Nelements, const int32_t offset, const int32_t* __restrict__ elementList,
    const G* __restrict__ ggeo, const T* __restrict__ D, const G* __restrict__ lambda, const T* __restrict__ q,
    T* __restrict__ Aq, const int* __restrict__ skip)
{
  using S = AxShape<T, NQ, BK, G>;
  constexpr bool EARLY = NF == 1 && S::early;
  using LL = LineLayout<T, NQ>;
  constexpr int NQ2 = NQ * NQ, NP = NQ2 * NQ, EPB = S::epb;
  if (skip && *skip) return;
  __shared__ T s_r[EPB][LL::SZ], s_s[EPB][LL::SS];
  const int t = threadIdx.x, slot = EPB > 1 ? (int)threadIdx.y : 0;
  int32_t block = blockIdx.x, f = 0;
  if constexpr (NF > 1) {
    const int32_t local = block >> 3;
    f = local % NF;
    block = (local / NF) * 8 + (block & 7);
    if ((int64_t)block * EPB >= Nelements) return;
  }
  const ElemPlace<PARTIAL, EPB> E(block * EPB, Nelements, elementList, slot);
  using IDX = typename ElemPlace<PARTIAL, EPB>::IDX;
  const IDX lo = E.rel * NP + t;
  GeoStream<T, NQ, BK, G, NF == 1, S::ahead, IDX> geo{ggeo + E.base * (int64_t)(kNggeo * NP), lambda + E.base * NP,
                                                      lambda + E.base * NP + offset, E.rel * (kNggeo * NP) + t, lo,
                                                      {}};
  const T* qf = q + E.base * NP + (int64_t)f * offset;
  T* Af = Aq + E.base * NP + (int64_t)f * offset;
  T rq[NQ], out[NQ];
#pragma unroll
  for (int k = 0; k < NQ; ++k) rq[k] = EARLY ? qf[lo + k * NQ2] : ldnt(&qf[lo + k * NQ2]);
  axhelm_lines<T, NQ, BK, false, EARLY>(
      t, rq, out, (ConstPtr<T>)D, s_r[slot], s_s[slot], geo, []() {},
      [&](T(&mq)[NQ]) {
#pragma unroll
        for (int k = 0; k < NQ; ++k) mq[k] = rq[k];
      });
  if (E.active) {
#pragma unroll
    for (int k = 0; k < NQ; ++k) stnt(out[k], &Af[lo + k * NQ2]);
  }
}

// Three fields in turn, the element's factors read once (GeoKept); the next
// field's q is loaded while the factors are applied to the current one.  Up to
// NQ = 6 the load is left out after the last field (12e6 nodes, with it / now:
// N = 2 FP64 Poisson 250 / 241 us, N = 5 FP64 Helmholtz 282 / 274, FP32 Poisson
// 108 / 104); above, the branch costs more than the load, whose lines the
// caches hold (1e6 nodes, FP64 Poisson: N = 8 31.9 us without the branch, 35.4
// with it, N = 9 22.8 / 24.5, N = 7 18.1 / 18.4).
template <typename T, int NQ, bool BK, bool PARTIAL, typename G>
__global__ __launch_bounds__((NQ * NQ * AxKept<T, NQ, BK>::epb), (AxKept<T, NQ, BK>::waves)) void k_axhelm_kept(
    const int32_t Nelements, const int32_t offset, const int32_t* __restrict__ elementList,
    const G* __restrict__ ggeo, const T* __restrict__ D, const G* __restrict__ lambda, const T* __restrict__ q,
    T* __restrict__ Aq, const int* __restrict__ skip)
{
  using LL = LineLayout<T, NQ>;
  constexpr int NF = 3, NQ2 = NQ * NQ, NP = NQ2 * NQ, EPB = AxKept<T, NQ, BK>::epb;
  if (skip && *skip) return;
  __shared__ T s_r[EPB][LL::SZ], s_s[EPB][LL::SS], s_l[BK ? 1 : EPB * NP], s_w[BK ? 1 : EPB * NP];
  const int t = threadIdx.x, slot = EPB > 1 ? (int)threadIdx.y : 0;
  const ElemPlace<PARTIAL, EPB> E((int32_t)blockIdx.x * EPB, Nelements, elementList, slot);
  using IDX = typename ElemPlace<PARTIAL, EPB>::IDX;
  const IDX lo = E.rel * NP + t;
  const T* qf = q + E.base * NP;
  T* Af = Aq + E.base * NP;
  T rq[NQ], out[NQ];
#pragma unroll
  for (int k = 0; k < NQ; ++k) rq[k] = ldnt(&qf[lo + k * NQ2]);
  GeoKept<T, NQ, BK, G, IDX> geo{{ggeo + E.base * (int64_t)(kNggeo * NP), lambda + E.base * NP,
                                  lambda + E.base * NP + offset, E.rel * (kNggeo * NP) + t, lo, {}},
                                 s_l + (BK ? 0 : slot * NP + t),
                                 s_w + (BK ? 0 : slot * NP + t)};
  geo.load();
#pragma unroll 1
  for (int f = 0; f < NF; ++f) {
    const T* qc = qf;
    if (f + 1 < NF) qf += offset;
    axhelm_lines<T, NQ, BK>(
        t, rq, out, (ConstPtr<T>)D, s_r[slot], s_s[slot], geo,
        [&]() {
          if (NQ > 6 || f + 1 < NF) {  // (at the end of NQ > 6 the last field's again, unused)
#pragma unroll
            for (int k = 0; k < NQ; ++k) rq[k] = qf[lo + k * NQ2];
          }
        },
        [&](T(&mq)[NQ]) {
          if (!BK) {
#pragma unroll
            for (int k = 0; k < NQ; ++k) mq[k] = qc[lo + k * NQ2];
          }
        });
    if (E.active) {
#pragma unroll
      for (int k = 0; k < NQ; ++k) stnt(out[k], &Af[lo + k * NQ2]);
    }
    Af += offset;
  }
}

// The three-field Helmholtz PCG form at 8 <= Nq <= 12 (FP64 and FP32
// geometry) sums a lane's share of pAp per field, then (f0 + f1) + f2; every
// other form runs one chain over fields then k.  The oracle states both.
template <int NQ, int NF, bool BK, typename G>
struct AxFieldSums {
  static constexpr bool value = NF == 3 && !BK && NQ >= 8 && NQ <= 12 && sizeof(G) != 2;
};

// Where the lane sums run per field, the fields can have a workgroup each and
// hand them on through memory (one value per line and field, 1 / Nq of a
// field, and a small kernel).  Small workgroups of two or three waves then
// take the place of one that holds three fields' lines in LDS or one field's
// registers on one wave per SIMD, and G and lambda of the fields after the
// first come from the XCD's L2.  us, the better other form / this one:
//            1e5 nodes      3e5            1e6            8e6
//   N = 9    11.3 / 11.0    22.3 / 16.3    46.5 / 38.3    365 / 307   FP64
//   N = 10   13.7 / 10.5    16.3 / 16.2    46.8 / 39.3    380 / 295   FP64
//   N = 11   14.7 / 11.5    17.7 / 20.1    50.6 / 42.5    355 / 314   FP64
//   N = 9    8.8 / 9.5      12.4 / 11.9    34.8 / 30.1    230 / 220   FP32
//   N = 10   10.5 / 9.5     11.7 / 12.2    36.0 / 29.9    266 / 218   FP32
//   N = 11   11.1 / 10.3    12.3 / 14.9    37.9 / 31.3    246 / 207   FP32
// N = 7 and 8 lose but for the smallest meshes, the small kernel not counted
// (FP64 at 8e6 nodes 202 / 261 and 274 / 348).  Where three workgroups an element no longer have a
// CU each, and up to one element a CU, only FP64 N = 9 and 10 gain.
template <int NQ, int NF, bool BK, typename T, typename G>
struct AxFieldBlocks {
  static constexpr bool value = AxFieldSums<NQ, NF, BK, G>::value && NQ >= 10;
  static constexpr bool always = value && sizeof(T) == 8 && NQ <= 11;
  static bool when(int64_t Nelements) { return always || Nelements >= 256 || 3 * Nelements <= 256; }
};

template <int NQ2>
constexpr int kTreeWidth = NQ2 <= 4 ? 4 : NQ2 <= 16 ? 16 : NQ2 <= 32 ? 32 : NQ2 <= 64 ? 64 : NQ2 <= 128 ? 128 : 256;

// Sum of the NQ2 lane values of an element in the halving tree over the next
// power of two (zero padded); valid in the slot's lane t = 0.  tid: the lane
// in the workgroup, slot 0's lanes first; `on` is false in lanes that take no
// part (every lane of the workgroup calls, for the barriers).
template <int NQ2, int EPB>
__device__ __forceinline__ double lane_tree(double v, double* s_red, const int slot, const int t, const int tid,
                                            const bool on)
{
  constexpr int P2 = kTreeWidth<NQ2>;
  if constexpr (P2 == NQ2 && P2 <= 64) {  // the slot's lanes are one aligned part of a wave
#pragma unroll
    for (int h = P2 / 2; h >= 1; h >>= 1) v += __shfl_xor(v, h, 64);
    return v;
  } else {
    double* const red = s_red + slot * P2;
    if (on) {
      red[t] = v;
      if (t + NQ2 < P2) red[t + NQ2] = 0.0;
    }
    if constexpr (P2 > 64) {
      // the first wave of each slot (EPB = 1 here) sums 64 lanes from registers
      static_assert(EPB == 1, "one element per workgroup from Nq = 9 up");
      __syncthreads();
      double x = 0.0;
      if (tid < 64) {
        x = P2 == 256 ? (red[tid] + red[tid + 128]) + (red[tid + 64] + red[tid + 192]) : red[tid] + red[tid + 64];
        x = wave_sum(x);
      }
      return x;
    } else {
      for (int h = P2 / 2; h >= 1; h >>= 1) {
        __syncthreads();
        if (on && t < h) red[t] = red[t] + red[t + h];
      }
      return red[0];
    }
  }
}

// PCG form (FP64): p = z + beta p (BPScaledAdd, nekBone/solve.cpp:100), then
// Ap_local = A p, and the element's share of pAp = sum_nodes p * Ap_local.
// Because p is continuous and zero on the mask, sum_local p (A_L p) equals
// <p, gs(A_L p)>_w exactly in real arithmetic (the weights 1/multiplicity
// undo the gather-scatter); this value is what BPAxOperator's dot returns.
// The lanes' shares are summed by lane_tree; the element partials go to
// partials[e].
// Three fields: in turn, one thread group of NQ2 lanes per field of an element
// (threadIdx.y = field; the groups hand the lane sums on through LDS in field
// order), or one workgroup per field (its lane sums go to memory; k_field_sums).
enum PcgFields { kInTurn, kGroups, kBlocks };
template <int NQ, int NF, bool BK, typename T, typename G, int FORM>
struct AxPcg {
  static constexpr bool kept = NF == 3 && FORM == kInTurn && AxKept<T, NQ, BK>::value;
  static constexpr int epb = FORM != kInTurn ? 1 : kept ? AxKept<T, NQ, BK>::epb : AxShape<T, NQ, BK>::epb;
  static constexpr int waves = kept ? AxKept<T, NQ, BK>::waves : 1;
  // the next field's z and p in flight during the current one, where the
  // registers allow it (after the last field nothing is loaded: 13824 elements,
  // 12 iterations FP64, with / without that load, N = 7 6.49 / 6.36 ms, N = 5
  // 3.04 / 2.99)
  static constexpr bool prefetch = kept && (sizeof(T) == 4 || NQ <= 8);
  static constexpr bool late = NF == 3 && FORM == kInTurn && !prefetch;
};

template <int NQ, int NF, bool BK, typename T, typename G, int FORM>
__global__ __launch_bounds__((NQ * NQ * AxPcg<NQ, NF, BK, T, G, FORM>::epb * (FORM == kGroups ? NF : 1)), (AxPcg<NQ, NF, BK, T, G, FORM>::waves)) void k_axhelm_pcg(
    const int32_t Nelements, const int32_t offset, const G* __restrict__ ggeo, const T* __restrict__ D,
    const G* __restrict__ lambda, const double* __restrict__ z, double* __restrict__ p, double* __restrict__ Ap,
    double* __restrict__ partials, double* __restrict__ lane_sums, const PcgFlags* __restrict__ S)
{
  using P = AxPcg<NQ, NF, BK, T, G, FORM>;
  constexpr bool FG = FORM == kGroups, FB = FORM == kBlocks;
  using LL = LineLayout<T, NQ>;
  constexpr bool SUMS = AxFieldSums<NQ, NF, BK, G>::value;
  constexpr int NQ2 = NQ * NQ, NP = NQ2 * NQ, EPB = P::epb, GR = EPB * (FG ? NF : 1), LOOP = FORM == kInTurn ? NF : 1;
  if (S->done) return;
  const double beta = S->beta;
  __shared__ T s_r[GR][LL::SZ], s_s[GR][LL::SS];
  __shared__ T s_l[P::kept && !BK ? EPB * NP : 1], s_w[P::kept && !BK ? EPB * NP : 1];
  __shared__ double s_red[EPB * kTreeWidth<NQ2>], s_acc[FG ? NF : 1][FG ? NQ2 : 1];
  const int t = threadIdx.x, y = GR > 1 ? (int)threadIdx.y : 0, slot = FG ? 0 : y;
  int32_t block = blockIdx.x;
  int field0 = FG ? y : 0;
  if constexpr (FB) {  // as k_axhelm: an element's fields follow each other on one XCD
    const int32_t local = block >> 3;
    field0 = local % NF;
    block = (local / NF) * 8 + (block & 7);
    if (block >= Nelements) return;
  }
  const ElemPlace<false, EPB> E(block * EPB, Nelements, nullptr, slot);
  const int32_t lo = E.rel * NP + t;
  const double* zf = z + E.base * NP + (int64_t)field0 * offset;
  double* pf = p + E.base * NP + (int64_t)field0 * offset;
  double* Af = Ap + E.base * NP + (int64_t)field0 * offset;
  const G* const gb = ggeo + E.base * (int64_t)(kNggeo * NP);
  const G* const lb = lambda + E.base * NP;
  const int32_t go = E.rel * (kNggeo * NP) + t;
  double zn[NQ], pn[NQ], acc = 0.0, fsum[NF];
  auto load_zp = [&]() {
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      pn[k] = pf[lo + k * NQ2];
      zn[k] = ldnt(&zf[lo + k * NQ2]);
    }
  };
  if (P::prefetch) load_zp();
  auto run = [&](auto& geo) {
#pragma unroll 1
    for (int f = 0; f < LOOP; ++f) {
      T rq[NQ], out[NQ];
      double pk[NQ];
      if (!P::prefetch) load_zp();
#pragma unroll
      for (int k = 0; k < NQ; ++k) {
        const double v = __builtin_fma(beta, pn[k], zn[k]);
        rq[k] = (T)v;
        if (E.active) pf[lo + k * NQ2] = v;
        if (LOOP == 1) pk[k] = v;
      }
      const double* const pc = pf;
      if (f + 1 < LOOP) {
        pf += offset;
        zf += offset;
      }
      axhelm_lines<T, NQ, BK, P::late>(
          t, rq, out, (ConstPtr<T>)D, s_r[y], s_s[y], geo,
          [&]() {
            if (P::prefetch && f + 1 < LOOP) load_zp();  // the next field's
          },
          [&](T(&mq)[NQ]) {
#pragma unroll
            for (int k = 0; k < NQ; ++k) {
              if (LOOP > 1) pk[k] = pc[lo + k * NQ2];  // this lane's own store
              mq[k] = (T)pk[k];
            }
          });
      if (SUMS) acc = 0.0;
      if constexpr (FG && !SUMS) {  // the chain over fields then k: each group continues the previous one's
        for (int c = 0; c < NF; ++c) {
          if (c == y) {
            acc = c == 0 ? 0.0 : s_acc[c - 1][t];
#pragma unroll
            for (int k = 0; k < NQ; ++k) acc = __builtin_fma(pk[k], (double)out[k], acc);
            s_acc[c][t] = acc;
          }
          __syncthreads();
        }
        acc = s_acc[NF - 1][t];
      } else {
#pragma unroll
        for (int k = 0; k < NQ; ++k) acc = __builtin_fma(pk[k], (double)out[k], acc);
      }
      if (E.active) {
#pragma unroll
        for (int k = 0; k < NQ; ++k) stnt((double)out[k], &Af[lo + k * NQ2]);
      }
      Af += offset;
      if (SUMS && FORM == kInTurn) {
        if (f == 0) fsum[0] = acc;
        else if (f == 1) fsum[NF > 1 ? 1 : 0] = acc;
        else fsum[NF - 1] = acc;
      }
    }
  };
  if constexpr (P::kept) {
    GeoKept<T, NQ, BK, G, int32_t> geo{{gb, lb, lb + offset, go, lo, {}},
                                       s_l + (BK ? 0 : slot * NP + t),
                                       s_w + (BK ? 0 : slot * NP + t)};
    geo.load();
    run(geo);
  } else {
    GeoStream<T, NQ, BK, G, NF == 1, AxShape<T, NQ, BK>::ahead, int32_t> geo{gb, lb, lb + offset, go, lo, {}};
    run(geo);
  }
  if constexpr (FB) {
    lane_sums[(E.base * NF + field0) * NQ2 + t] = acc;
    return;
  }
  if constexpr (SUMS && FG) {
    s_acc[y][t] = acc;
    __syncthreads();
    acc = (s_acc[0][t] + s_acc[1][t]) + s_acc[2][t];
  } else if constexpr (SUMS && FORM == kInTurn) {
    acc = (fsum[0] + fsum[1]) + fsum[2];
  }
  const double sum = lane_tree<NQ2, EPB>(acc, s_red, slot, t, y * NQ2 + t, y == slot);
  if (t == 0 && y == slot && E.active) partials[E.base + E.rel] = sum;
}

// partials[e] of the one-workgroup-per-field form: (f0 + f1) + f2 per lane,
// then lane_tree's order; a wave per element.  Launch-bound (about 2.5 us at
// 1e6 nodes).
template <int NQ2>
__global__ __launch_bounds__(256) void k_field_sums(const int32_t Nelements, const double* __restrict__ lane_sums,
                                                    double* __restrict__ partials, const PcgFlags* __restrict__ S)
{
  constexpr int P2 = kTreeWidth<NQ2>;
  static_assert(P2 == 128 || P2 == 256, "two or four values a lane");
  if (S->done) return;
  const int l = threadIdx.x & 63;
  const int64_t e = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (e >= Nelements) return;
  const double* const a = lane_sums + e * 3 * NQ2;
  double v[P2 / 64];
#pragma unroll
  for (int u = 0; u < P2 / 64; ++u) {
    const int t = l + 64 * u;
    v[u] = t < NQ2 ? (a[t] + a[NQ2 + t]) + a[2 * NQ2 + t] : 0.0;
  }
  const double x = wave_sum(P2 == 256 ? (v[0] + v[P2 / 128]) + (v[1] + v[P2 / 64 - 1]) : v[0] + v[1]);
  if (l == 0) partials[e] = x;
}

// Local Jacobi diagonal, nekBone/kernel/updateJacobi.okl:27-108, same
// expression order as the reference (plain mul/add, no contraction): the
// products G lambda0 of the three directions are formed once per node, in LDS,
// where every node of their line reads them (each lane had loaded 3 Nq factors
// and lambda values a node; 32768 elements, N = 7: 544 -> 255 us).
template <int NQ>
__global__ __launch_bounds__(NQ* NQ) void k_jacobi(const int32_t Nelements, const int32_t offset,
                                                   const int32_t* __restrict__ mapB,
                                                   const double* __restrict__ ggeo,
                                                   const double* __restrict__ D,
                                                   const double* __restrict__ lambda,
                                                   double* __restrict__ diag)
{
  constexpr int NQ2 = NQ * NQ;
  constexpr int NP = NQ2 * NQ;
  __shared__ double s_D[NQ2], s_g[3][NP];
  const int t = threadIdx.x, i = t % NQ, j = t / NQ;
  const int64_t e = blockIdx.x;
  const double* g = ggeo + e * (int64_t)(kNggeo * NP);
  const double* l0 = lambda + e * NP;
  s_D[t] = D[t];
#pragma unroll
  for (int k = 0; k < NQ; ++k) {
    const int n = t + k * NQ2;
    const double lambda_0 = l0[n];
    s_g[0][n] = ldnt(&g[kG00 * NP + n]) * lambda_0;
    s_g[1][n] = ldnt(&g[kG11 * NP + n]) * lambda_0;
    s_g[2][n] = ldnt(&g[kG22 * NP + n]) * lambda_0;
  }
  __syncthreads();
  const double Dii = s_D[i * NQ + i], Djj = s_D[j * NQ + j];
#pragma unroll 2
  for (int k = 0; k < NQ; ++k) {
    const int n = t + k * NQ2;
    const int64_t id = e * NP + n;
    const double Dkk = s_D[k * NQ + k], lambda_0 = l0[n];
    double r_q = 0.0;
    r_q += 2.0 * ldnt(&g[kG01 * NP + n]) * lambda_0 * Dii * Djj;
    r_q += 2.0 * ldnt(&g[kG02 * NP + n]) * lambda_0 * Dii * Dkk;
    r_q += 2.0 * ldnt(&g[kG12 * NP + n]) * lambda_0 * Djj * Dkk;
#pragma unroll
    for (int m = 0; m < NQ; ++m) {
      const double Di = s_D[m * NQ + i], Dj = s_D[m * NQ + j], Dk = s_D[m * NQ + k];
      r_q += s_g[0][m + j * NQ + k * NQ2] * Di * Di;
      r_q += s_g[1][i + m * NQ + k * NQ2] * Dj * Dj;
      r_q += s_g[2][t + m * NQ2] * Dk * Dk;
    }
    r_q += ldnt(&g[kGWJ * NP + n]) * ldnt(&lambda[id + offset]);
    diag[id] = mapB && mapB[id] == 1 ? 1.0 : r_q;
  }
}

template <typename T, int NQ, int NF, bool BK, bool PARTIAL, typename G = T>
static int launch_axhelm_t(int32_t Nelements, int32_t offset, const int32_t* elementList,
                           const void* ggeo, const void* D, const void* lambda, const void* q, void* Aq,
                           const int* skip, hipStream_t s)
{
  if (Nelements <= 0) return NBX_SUCCESS;
  if constexpr (NF == 3 && AxKept<T, NQ, BK>::value) {
    if (AxKept<T, NQ, BK>::when(Nelements)) {
      constexpr int EPB = AxKept<T, NQ, BK>::epb;
      hipLaunchKernelGGL((k_axhelm_kept<T, NQ, BK, PARTIAL, G>), dim3((Nelements + EPB - 1) / EPB),
                         dim3(NQ * NQ, EPB), 0, s, Nelements, offset, elementList, (const G*)ggeo, (const T*)D,
                         (const G*)lambda, (const T*)q, (T*)Aq, skip);
      NBX_HIP_LAUNCH();
      return NBX_SUCCESS;
    }
  }
  constexpr int EPB = AxShape<T, NQ, BK>::epb;
  const int32_t blocks = (Nelements + EPB - 1) / EPB;
  const unsigned grid = NF == 1 ? (unsigned)blocks : (unsigned)((blocks + 7) / 8 * 8) * NF;
  hipLaunchKernelGGL((k_axhelm<T, NQ, NF, BK, PARTIAL, G>), dim3(grid), dim3(NQ * NQ, EPB), 0, s, Nelements, offset,
                     elementList, (const G*)ggeo, (const T*)D, (const G*)lambda, (const T*)q, (T*)Aq, skip);
  NBX_HIP_LAUNCH();
  return NBX_SUCCESS;
}

template <typename T, int NQ, typename G = T>
static int dispatch_flags(int Nf, int bk, bool partial, int32_t Nelements, int32_t offset,
                          const int32_t* elementList, const void* ggeo, const void* D,
                          const void* lambda, const void* q, void* Aq, const int* skip, hipStream_t s)
{
  if (!std::is_same<T, G>::value) {  // bf16 geometry: one field, whole mesh
    if (Nf != 1 || partial) return fail(NBX_ERR_UNSUPPORTED, "axhelm bf16: one field, no element list");
    if (bk) return launch_axhelm_t<T, NQ, 1, true, false, G>(Nelements, offset, nullptr, ggeo, D, lambda, q, Aq, skip, s);
    return launch_axhelm_t<T, NQ, 1, false, false, G>(Nelements, offset, nullptr, ggeo, D, lambda, q, Aq, skip, s);
  } else {
#define NBX_AX_CASE(NFV, BKV, PV)                                                               \
  if (Nf == NFV && (bk != 0) == BKV && partial == PV)                                           \
    return launch_axhelm_t<T, NQ, NFV, BKV, PV>(Nelements, offset, elementList, ggeo, D, lambda, \
                                                 q, Aq, skip, s);
  NBX_AX_CASE(1, false, false)
  NBX_AX_CASE(1, true, false)
  NBX_AX_CASE(3, false, false)
  NBX_AX_CASE(3, true, false)
  NBX_AX_CASE(1, false, true)
  NBX_AX_CASE(1, true, true)
  NBX_AX_CASE(3, false, true)
  NBX_AX_CASE(3, true, true)
#undef NBX_AX_CASE
  }
  return fail(NBX_ERR_UNSUPPORTED, "axhelm: Nfields=%d not supported (1 or 3)", Nf);
}

template <typename T, typename G = T>
static int dispatch_n(int N, int Nf, int bk, bool partial, int32_t Nelements, int32_t offset,
                      const int32_t* elementList, const void* ggeo, const void* D, const void* lambda,
                      const void* q, void* Aq, const int* skip, hipStream_t s)
{
  switch (N) {
#define NBX_N_CASE(NV) \
  case NV:             \
    return dispatch_flags<T, NV + 1, G>(Nf, bk, partial, Nelements, offset, elementList, ggeo, D, lambda, q, Aq, skip, s);
    NBX_N_CASE(1)
    NBX_N_CASE(2)
    NBX_N_CASE(3)
    NBX_N_CASE(4)
    NBX_N_CASE(5)
    NBX_N_CASE(6)
    NBX_N_CASE(7)
    NBX_N_CASE(8)
    NBX_N_CASE(9)
    NBX_N_CASE(10)
    NBX_N_CASE(11)
    NBX_N_CASE(12)
    NBX_N_CASE(13)
    NBX_N_CASE(14)
    NBX_N_CASE(15)
#undef NBX_N_CASE
    default:
      return fail(NBX_ERR_UNSUPPORTED, "axhelm: N=%d not supported (1..15)", N);
  }
}

template <int NQ, int NF, bool BK, typename T, typename G>
static void axhelm_pcg_launch_k(int32_t Nelements, int32_t offset, const void* ggeo, const void* D,
                                const void* lambda, const double* z, double* p, double* Ap, double* partials,
                                double* lane_sums, const PcgFlags* S, hipStream_t s)
{
  if constexpr (AxFieldBlocks<NQ, NF, BK, T, G>::value) {
    if (AxFieldBlocks<NQ, NF, BK, T, G>::when(Nelements)) {
      hipLaunchKernelGGL((k_axhelm_pcg<NQ, NF, BK, T, G, kBlocks>), dim3((unsigned)((Nelements + 7) / 8 * 8) * NF),
                         dim3(NQ * NQ), 0, s, Nelements, offset, (const G*)ggeo, (const T*)D, (const G*)lambda, z, p,
                         Ap, partials, lane_sums, S);
      hipLaunchKernelGGL(k_field_sums<NQ * NQ>, dim3((Nelements + 3) / 4), dim3(256), 0, s, Nelements, lane_sums,
                         partials, S);
      return;
    }
  }
  if constexpr (NF == 3 && AxFieldGroups<T, NQ, BK, G>::fits && !AxFieldBlocks<NQ, NF, BK, T, G>::always) {
    if (AxFieldGroups<T, NQ, BK, G>::when(Nelements)) {
      hipLaunchKernelGGL((k_axhelm_pcg<NQ, NF, BK, T, G, kGroups>), dim3(Nelements), dim3(NQ * NQ, NF), 0, s,
                         Nelements, offset, (const G*)ggeo, (const T*)D, (const G*)lambda, z, p, Ap, partials,
                         lane_sums, S);
      return;
    }
  }
  if constexpr (!AxFieldBlocks<NQ, NF, BK, T, G>::always && !(NF == 3 && AxFieldGroups<T, NQ, BK, G>::always)) {
    constexpr int EPB = AxPcg<NQ, NF, BK, T, G, kInTurn>::epb;
    hipLaunchKernelGGL((k_axhelm_pcg<NQ, NF, BK, T, G, kInTurn>), dim3((Nelements + EPB - 1) / EPB),
                       dim3(NQ * NQ, EPB), 0, s, Nelements, offset, (const G*)ggeo, (const T*)D, (const G*)lambda, z,
                       p, Ap, partials, lane_sums, S);
  }
}

template <typename T, typename G>
static int axhelm_pcg_launch_t(int N, int Nf, int bk, int32_t Nelements, int32_t offset, const void* ggeo,
                               const void* D, const void* lambda, const double* z, double* p, double* Ap,
                               double* partials, double* lane_sums, const PcgFlags* S, hipStream_t s)
{
#define NBX_AXP(NV)                                                                                              \
  case NV:                                                                                                       \
    if (Nelements < 1) break;                                                                                    \
    if (Nf == 1 && bk)                                                                                           \
      axhelm_pcg_launch_k<NV + 1, 1, true, T, G>(Nelements, offset, ggeo, D, lambda, z, p, Ap, partials,           \
                                                   lane_sums, S, s);                                            \
    else if (Nf == 1)                                                                                            \
      axhelm_pcg_launch_k<NV + 1, 1, false, T, G>(Nelements, offset, ggeo, D, lambda, z, p, Ap, partials,           \
                                                   lane_sums, S, s);                                            \
    else if (bk)                                                                                                 \
      axhelm_pcg_launch_k<NV + 1, 3, true, T, G>(Nelements, offset, ggeo, D, lambda, z, p, Ap, partials,           \
                                                   lane_sums, S, s);                                            \
    else                                                                                                         \
      axhelm_pcg_launch_k<NV + 1, 3, false, T, G>(Nelements, offset, ggeo, D, lambda, z, p, Ap, partials,           \
                                                   lane_sums, S, s);                                            \
    break;
  if (Nf != 1 && Nf != 3) return fail(NBX_ERR_UNSUPPORTED, "axhelm_pcg: Nfields=%d", Nf);
  switch (N) {
    NBX_AXP(1)
    NBX_AXP(2)
    NBX_AXP(3)
    NBX_AXP(4)
    NBX_AXP(5)
    NBX_AXP(6)
    NBX_AXP(7)
    NBX_AXP(8)
    NBX_AXP(9)
    NBX_AXP(10)
    NBX_AXP(11)
    NBX_AXP(12)
    NBX_AXP(13)
    NBX_AXP(14)
    NBX_AXP(15)
    default:
      return fail(NBX_ERR_UNSUPPORTED, "axhelm_pcg: N=%d", N);
  }
#undef NBX_AXP
  NBX_HIP_LAUNCH();
  return NBX_SUCCESS;
}


// per-precision entry points of the dispatch (one translation unit each)
int axhelm_dispatch_f64(int N, int Nf, int bk, bool partial, int32_t Nelements, int32_t offset,
                        const int32_t* elementList, const void* ggeo, const void* D, const void* lambda,
                        const void* q, void* Aq, const int* skip, hipStream_t s);
int axhelm_dispatch_f32(int N, int Nf, int bk, bool partial, int32_t Nelements, int32_t offset,
                        const int32_t* elementList, const void* ggeo, const void* D, const void* lambda,
                        const void* q, void* Aq, const int* skip, hipStream_t s);
int axhelm_dispatch_bf16(int N, int Nf, int bk, bool partial, int32_t Nelements, int32_t offset,
                         const int32_t* elementList, const void* ggeo, const void* D, const void* lambda,
                         const void* q, void* Aq, const int* skip, hipStream_t s);
int axhelm_pcg_dispatch_f64(int N, int Nf, int bk, int32_t Nelements, int32_t offset, const void* ggeo,
                            const void* D, const void* lambda, const double* z, double* p, double* Ap,
                            double* partials, double* lane_sums, const PcgFlags* S, hipStream_t s);
int axhelm_pcg_dispatch_f32(int N, int Nf, int bk, int32_t Nelements, int32_t offset, const void* ggeo,
                            const void* D, const void* lambda, const double* z, double* p, double* Ap,
                            double* partials, double* lane_sums, const PcgFlags* S, hipStream_t s);
int axhelm_pcg_dispatch_bf16(int N, int Nf, int bk, int32_t Nelements, int32_t offset, const void* ggeo,
                             const void* D, const void* lambda, const double* z, double* p, double* Ap,
                             double* partials, double* lane_sums, const PcgFlags* S, hipStream_t s);

}  // namespace nbx
