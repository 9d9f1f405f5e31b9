// axhelm with the tensor contractions on the matrix cores: bf16 or fp16
// operands, FP32 accumulation (v_mfma_f32_16x16x16_bf16 / _f16), N = 7 and 9,
// one or three fields.  The geometric factors are applied in FP32 on the
// vector ALUs exactly as in the FP32 kernel:
//
//   q_h  = h(q),  D_h = h(D)            h = round to the operand type (nearest even)
//   qr   = D_h q_h along r (FP32 accumulate), qs, qt alike
//   Gr   = fma(G02, qt, fma(G01, qs, G00 qr))  (and Gs, Gt), non-BK * lambda0
//   Aq   = D_h^T h(Gr) + D_h^T h(Gs) + D_h^T h(Gt)   (summed r, s, t)
//          non-BK: + GWJ lambda1 q
//
// MFMA lane layout (16x16x16): lane l holds A[l%16][4(l/16)+i],
// B[4(l/16)+i][l%16] and C[4(l/16)+i][l%16], i = 0..3.
// bf16 keeps the FP32 exponent range, so small residuals do not underflow;
// fp16 carries 3 more significand bits but its normal range ends at 2^-14,
// so it serves operands of order one (the geometric factors stay FP32: on
// fine meshes GWJ falls below that range).
#include "nbx_internal.h"

namespace nbx {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// v_cvt_pk_bf16_f32: nearest even, the bits of bf16_bits for every non-NaN input
__device__ __forceinline__ short f2bf(float x) { return (short)bf16_bits_hw(x); }

// matrix-core operand types: storage element, 4-vector, rounding, product
struct OpBf16 {
  typedef short elem;
  typedef short vec4 __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ elem round(float x) { return f2bf(x); }
  static __device__ __forceinline__ f32x4 mma(const vec4& a, const vec4& b, const f32x4& c)
  {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
  }
};

struct OpF16 {
  typedef _Float16 elem;
  typedef _Float16 vec4 __attribute__((ext_vector_type(4)));
  // v_cvt_f16_f32: nearest even, fp16 subnormals kept
  static __device__ __forceinline__ elem round(float x) { return (_Float16)x; }
  static __device__ __forceinline__ f32x4 mma(const vec4& a, const vec4& b, const f32x4& c)
  {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(a, b, c, 0, 0, 0);
  }
};

// two neighbouring values at the element type's alignment
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2a __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t u32a2 __attribute__((aligned(2)));
__device__ __forceinline__ f32x2 ld2(const float* p)
{
  return __builtin_nontemporal_load(reinterpret_cast<const f32x2a*>(p));
}
__device__ __forceinline__ f32x2 ld2(const uint16_t* p)
{
  const uint32_t v = __builtin_nontemporal_load(reinterpret_cast<const u32a2*>(p));
  return f32x2{__uint_as_float(v << 16), __uint_as_float(v & 0xffff0000u)};
}

// One element per workgroup, two nodes (neighbours in r) per lane, the fields
// in turn; each 1-D contraction of a field is a (16 x 16) by (16 x Nq^2) product
// with D zero-padded to 16 x 16, columns in tiles of 16 (padded rows multiply
// zeros, padded columns and output rows are never read).
//
// Bound by LDS traffic and the four barriers a field, so the layouts keep both
// the wave count and the bank conflicts in hand:
// - operands: for direction d the column c runs over the other two indices and
//   the contracted index is contiguous, so a lane's four operands are one
//   8-byte read.  A column keeps its 10 (8) rows, not 16: lanes of the last
//   rows feed zeros from registers.
// - products: D B for r, whose rows are then contiguous per column, and
//   (B^T D^T), the same registers with the operands exchanged, for s and t,
//   whose columns are contiguous per row; either way a lane writes its four
//   products at once and a node pair is read back with one 8-byte read.
// 24 KB (N = 9) and two nodes a lane leave room for eight waves per SIMD.
// The next field's q is in flight during the current one; geometry and lambda
// are read once per element.
//
// 8e6 nodes, us, against one 256-lane workgroup per element with four nodes a
// lane and columns of 20 entries (40 KB), and at N = 7 with one field one wave
// per element pair:
//   bf16 geometry, Helmholtz  N = 9  three fields 140 -> 91 (3.7 TB/s), one 75 -> 47
//                             N = 7  three fields 114 -> 81,            one 81 -> 43
//   fp16 operands, Poisson    N = 9  three fields 139 -> 94,            one 72 -> 51
template <int NQ>
struct Mma16 {
  static constexpr int NQ2 = NQ * NQ, P = NQ2 * NQ, CT = (NQ2 + 15) / 16, NC = CT * 16;
  static constexpr int OWN = P / 2;  // a lane owns two neighbours in r
  static constexpr int TH = (OWN + 63) / 64 * 64, WAVES = TH / 64;
  static constexpr int R = (NQ + 3) / 4 * 4;  // rows kept of a column: whole groups of four
  static constexpr int BS = 12;               // r, s operand column stride: 24 bytes, aligned 8-byte reads
  static constexpr int BT = 14;               // t operand column stride: 7 banks
  static constexpr int RS = R;                // r product column stride: aligned 16-byte writes
  static constexpr int ST = NQ == 8 ? 72 : NC + 4;  // s, t product row stride
  static_assert((NQ == 8 || NQ == 10) && R <= BS, "rows of a column within its stride");
};

template <int NQ, int NF, bool BK, typename G, typename OP>
__global__ __launch_bounds__(Mma16<NQ>::TH, 8) void k_axhelm_mma16(
    const int32_t Nelements, const int32_t offset, const G* __restrict__ ggeo, const float* __restrict__ D,
    const G* __restrict__ lambda, const float* __restrict__ q, float* __restrict__ Aq, const int* __restrict__ skip)
{
  using M = Mma16<NQ>;
  constexpr int P = M::P, NQ2 = M::NQ2, CT = M::CT, NC = M::NC, OWN = M::OWN, BS = M::BS, BT = M::BT, RS = M::RS,
                ST = M::ST;
  typedef typename OP::elem H;
  typedef typename OP::vec4 V4;
  if (skip && *skip) return;
  __shared__ __align__(16) H s_b[NC * (2 * BS + BT)];  // operands per direction: h(q), then h(G)
  __shared__ __align__(16) float s_r[NC * RS], s_s[NQ * ST], s_t[NQ * ST];
  const int t = threadIdx.x, l = t & 63, w = t >> 6, kb = 4 * (l >> 4), lc = l & 15;
  const int64_t e = blockIdx.x;
  const float* qf = q + e * P;
  const bool on = OWN == M::TH || t < OWN;
  const int own = on ? t : OWN - 1;
  f32x2 qn = ld2(&qf[2 * own]);  // the next field's q, in flight during the current field
  // zero operands once: the padding rows (contracted index >= Nq) stay zero
  for (int u = t; u < NC * (2 * BS + BT) / 4; u += M::TH) reinterpret_cast<V4*>(s_b)[u] = V4{};
  V4 Af, At;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int k = kb + i;
    const bool in = lc < NQ && k < NQ;
    Af[i] = in ? OP::round(D[lc * NQ + k]) : (H)0;
    At[i] = in ? OP::round(D[k * NQ + lc]) : (H)0;
  }
  // this lane's nodes (i, j, k) and (i + 1, j, k): their places in the three
  // direction orders, and geometry
  const int i = 2 * (own % (NQ / 2)), j = (own / (NQ / 2)) % NQ, k = own / (NQ2 / 2);
  H* const b0 = &s_b[(j + NQ * k) * BS + i];
  H* const b1 = &s_b[(NC + i + NQ * k) * BS + j];
  H* const b2 = &s_b[2 * NC * BS + (i + NQ * j) * BT + k];
  const float* const c0 = &s_r[(j + NQ * k) * RS + i];
  const float* const c1 = &s_s[j * ST + i + NQ * k];
  const float* const c2 = &s_t[k * ST + i + NQ * j];
  f32x2 gf[6], l0, wl1;
  {
    const G* g = ggeo + e * (int64_t)(kNggeo * P) + 2 * own;
    const G* lam = lambda + e * P + 2 * own;
    gf[0] = ld2(&g[kG00 * P]);
    gf[1] = ld2(&g[kG01 * P]);
    gf[2] = ld2(&g[kG02 * P]);
    gf[3] = ld2(&g[kG11 * P]);
    gf[4] = ld2(&g[kG12 * P]);
    gf[5] = ld2(&g[kG22 * P]);
    l0 = wl1 = f32x2{1.f, 1.f};
    if (!BK) {
      l0 = ld2(lam);
      const f32x2 m = ld2(&g[kGWJ * P]), l1 = ld2(&lam[offset]);
      wl1 = f32x2{m[0] * l1[0], m[1] * l1[1]};
    }
  }
  // a (direction, column tile) product per wave turn
  auto products = [&](const V4& A) {
#pragma unroll
    for (int it = 0; it < (3 * CT + M::WAVES - 1) / M::WAVES; ++it) {
      const int tile = w + M::WAVES * it;
      if (tile >= 3 * CT) break;
      V4 B{};
      if (kb < NQ) {
        if (tile < 2 * CT) {
          B = *reinterpret_cast<const V4*>(&s_b[(tile * 16 + lc) * BS + kb]);
        } else {
          const uint32_t* const b =
              reinterpret_cast<const uint32_t*>(&s_b[2 * NC * BS + ((tile - 2 * CT) * 16 + lc) * BT + kb]);
          const uint32_t h[2] = {b[0], b[1]};
          B = __builtin_bit_cast(V4, h);
        }
      }
      if (tile < CT) {
        const f32x4 C = OP::mma(A, B, f32x4{0.f, 0.f, 0.f, 0.f});  // rows i of column lc
        if (kb < NQ) *reinterpret_cast<f32x4*>(&s_r[(tile * 16 + lc) * RS + kb]) = C;
      } else {
        const f32x4 C = OP::mma(B, A, f32x4{0.f, 0.f, 0.f, 0.f});  // columns kb .. kb + 3 of row lc
        float* const o = tile < 2 * CT ? s_s + (tile - CT) * 16 : s_t + (tile - 2 * CT) * 16;
        if (lc < NQ) *reinterpret_cast<f32x4*>(&o[lc * ST + kb]) = C;
      }
    }
  };
  __syncthreads();
  auto stage = [&](const f32x2& r, const f32x2& s, const f32x2& t) {
    const uint32_t lo = __builtin_bit_cast(uint16_t, OP::round(r[0])), hi = __builtin_bit_cast(uint16_t, OP::round(r[1]));
    *reinterpret_cast<uint32_t*>(b0) = lo | hi << 16;
    b1[0] = OP::round(s[0]);
    b1[BS] = OP::round(s[1]);
    b2[0] = OP::round(t[0]);
    b2[BT] = OP::round(t[1]);
  };
#pragma unroll 1
  for (int f = 0; f < NF; ++f) {
    const f32x2 qv = qn;
    if (on) stage(qv, qv, qv);
    if (f + 1 < NF) {
      qf += offset;
      qn = ld2(&qf[2 * own]);
    }
    __syncthreads();
    products(Af);
    __syncthreads();
    if (on) {
      const f32x2 qr = *reinterpret_cast<const f32x2*>(c0), qs = *reinterpret_cast<const f32x2*>(c1),
                  qt = *reinterpret_cast<const f32x2*>(c2);
      f32x2 Gr, Gs, Gt;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        Gr[u] = __builtin_fmaf(gf[2][u], qt[u], __builtin_fmaf(gf[1][u], qs[u], gf[0][u] * qr[u]));
        Gs[u] = __builtin_fmaf(gf[4][u], qt[u], __builtin_fmaf(gf[3][u], qs[u], gf[1][u] * qr[u]));
        Gt[u] = __builtin_fmaf(gf[5][u], qt[u], __builtin_fmaf(gf[4][u], qs[u], gf[2][u] * qr[u]));
        if (!BK) {
          Gr[u] = l0[u] * Gr[u];
          Gs[u] = l0[u] * Gs[u];
          Gt[u] = l0[u] * Gt[u];
        }
      }
      stage(Gr, Gs, Gt);
    }
    __syncthreads();
    products(At);
    __syncthreads();
    if (on) {
      const f32x2 r = *reinterpret_cast<const f32x2*>(c0), s = *reinterpret_cast<const f32x2*>(c1),
                  t = *reinterpret_cast<const f32x2*>(c2);
      f32x2 res;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        res[u] = (r[u] + s[u]) + t[u];
        if (!BK) res[u] = __builtin_fmaf(wl1[u], qv[u], res[u]);
      }
      __builtin_nontemporal_store(f32x2a(res), reinterpret_cast<f32x2a*>(&Aq[(int64_t)f * offset + e * P + 2 * own]));
    }
    // the next field's staging writes s_b only; its first barrier orders
    // these reads of the products before its own overwrite them
  }
}

int axhelm_mma_launch(int N, int Nf, int bk, bool f16_operands, int32_t Nelements, int32_t offset,
                      const void* ggeo, const void* D, const void* lambda, const void* q, void* Aq,
                      const int* skip, hipStream_t s)
{
  const char* name = f16_operands ? "axhelm fp16-MFMA" : "axhelm bf16-MFMA";
  if (!((N == 7 || N == 9) && (Nf == 1 || Nf == 3)))
    return fail(NBX_ERR_UNSUPPORTED, "%s: N = 7 or 9, one or three fields", name);
  if (Nelements <= 0) return Nelements == 0 ? NBX_SUCCESS : fail(NBX_ERR_INVALID, "axhelm: Nelements < 0");
  if (Nf == 3 && offset < Nelements * (N + 1) * (N + 1) * (N + 1))
    return fail(NBX_ERR_INVALID, "axhelm: offset < Nelements * Np");
#define NBX_MMA16(NQV, NFV, BKV, GT, OPT)                                                                         \
  hipLaunchKernelGGL((k_axhelm_mma16<NQV, NFV, BKV, GT, OPT>), dim3((unsigned)Nelements), dim3(Mma16<NQV>::TH), 0, \
                     s, Nelements, offset, (const GT*)ggeo, (const float*)D, (const GT*)lambda, (const float*)q,  \
                     (float*)Aq, skip)
#define NBX_MMA16_BK(NQV, NFV, GT, OPT) \
  if (bk) NBX_MMA16(NQV, NFV, true, GT, OPT); else NBX_MMA16(NQV, NFV, false, GT, OPT);
#define NBX_MMA16_T(NQV, NFV)                                   \
  if (f16_operands) { NBX_MMA16_BK(NQV, NFV, float, OpF16) }     \
  else { NBX_MMA16_BK(NQV, NFV, uint16_t, OpBf16) }
  if (N == 7 && Nf == 1) { NBX_MMA16_T(8, 1) }
  else if (N == 7) { NBX_MMA16_T(8, 3) }
  else if (Nf == 1) { NBX_MMA16_T(10, 1) }
  else { NBX_MMA16_T(10, 3) }
#undef NBX_MMA16_T
#undef NBX_MMA16_BK
#undef NBX_MMA16
  NBX_HIP_LAUNCH();
  return NBX_SUCCESS;
}

}  // namespace nbx
