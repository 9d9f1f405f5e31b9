// axhelm: tensor-product Helmholtz operator on hexahedral spectral elements.
//
// Reference semantics: axhelm/kernel/CPU/axhelm.c:27-413 (v0, n3_v0, bk_v0,
// bk_n3_v0), the Partial forms axhelm/kernel/VOLTA/axhelm.okl:158-290 and
// the host oracle axhelm/axhelmReference.cpp:19-101.
//
// Mapping to gfx950: Nq*Nq lanes per element (one wave64 at N=7, several
// elements per workgroup at small orders).  A lane owns a node column, an r
// line and an s line of the element in turn; lines are exchanged through LDS,
// the t direction stays in registers, and D's rows are scalar operands
// (axhelm_lines).  ggeo is streamed plane by plane, coalesced (64 consecutive
// doubles per load per factor at N=7).
//
// FP64 arithmetic order (identical to the CPU oracle, bit-exact):
//   qr = fma chain over m of D[i][m] q(m,j,k), qs and qt alike
//   Gqr = fma(G02,qt, fma(G01,qs, G00*qr)), Gqs, Gqt alike; non-BK * lambda0
//   Aq  = ((Aqr + Aqs) + Aqt), non-BK: fma(GWJ*lambda1, q, .)
#include "nbx_axhelm_impl.h"

namespace nbx {

int axhelm_dispatch_f64(int N, int Nf, int bk, bool partial, int32_t Nelements, int32_t offset,
                        const int32_t* elementList, const void* ggeo, const void* D, const void* lambda,
                        const void* q, void* Aq, const int* skip, hipStream_t s)
{
  return dispatch_n<double>(N, Nf, bk, partial, Nelements, offset, elementList, ggeo, D, lambda, q, Aq, skip, s);
}

int axhelm_pcg_dispatch_f64(int N, int Nf, int bk, int32_t Nelements, int32_t offset, const void* ggeo,
                            const void* D, const void* lambda, const double* z, double* p, double* Ap,
                            double* partials, double* lane_sums, const PcgFlags* S, hipStream_t s)
{
  return axhelm_pcg_launch_t<double, double>(N, Nf, bk, Nelements, offset, ggeo, D, lambda, z, p, Ap, partials,
                                            lane_sums, S, s);
}

int axhelm_launch(int N, int Nf, int bk, nbx_prec prec, int32_t Nelements, int32_t offset,
                  const int32_t* elementList, const void* ggeo, const void* D, const void* lambda,
                  const void* q, void* Aq, const int* skip, hipStream_t s)
{
  const bool partial = elementList != nullptr;
  switch (prec) {
    case NBX_F64:
      return axhelm_dispatch_f64(N, Nf, bk, partial, Nelements, offset, elementList, ggeo, D, lambda, q, Aq, skip,
                                 s);
    case NBX_F32:
      return axhelm_dispatch_f32(N, Nf, bk, partial, Nelements, offset, elementList, ggeo, D, lambda, q, Aq, skip,
                                 s);
    case NBX_BF16:  // FP32 vectors and arithmetic, bf16 geometric factors and lambda
      return axhelm_dispatch_bf16(N, Nf, bk, partial, Nelements, offset, elementList, ggeo, D, lambda, q, Aq,
                                  skip, s);
    case NBX_BF16_MFMA:  // as NBX_BF16 with the contractions on the matrix cores
      if (partial) return fail(NBX_ERR_UNSUPPORTED, "axhelm bf16-MFMA: no element list");
      return axhelm_mma_launch(N, Nf, bk, false, Nelements, offset, ggeo, D, lambda, q, Aq, skip, s);
    case NBX_F16:  // fp16 matrix-core operands, FP32 geometry, vectors and accumulation
      if (partial) return fail(NBX_ERR_UNSUPPORTED, "axhelm fp16-MFMA: no element list");
      return axhelm_mma_launch(N, Nf, bk, true, Nelements, offset, ggeo, D, lambda, q, Aq, skip, s);
    default:
      return fail(NBX_ERR_UNSUPPORTED, "axhelm: precision %d not supported by nbx_axhelm", (int)prec);
  }
}

// AxFieldBlocks, the union over the types
int64_t axhelm_pcg_lane_sums(int N, int Nf, int bk)
{
  return Nf == 3 && !bk && N >= 9 && N <= 11 ? 3 * (N + 1) * (N + 1) : 0;
}

int axhelm_pcg_launch(int N, int Nf, int bk, nbx_prec prec, int32_t Nelements, int32_t offset, const void* ggeo,
                      const void* D, const void* lambda, const double* z, double* p, double* Ap,
                      double* partials, double* lane_sums, const PcgFlags* S, hipStream_t s)
{
  switch (prec) {
    case NBX_F64:
      return axhelm_pcg_dispatch_f64(N, Nf, bk, Nelements, offset, ggeo, D, lambda, z, p, Ap, partials,
                                                 lane_sums, S, s);
    case NBX_F32:
      return axhelm_pcg_dispatch_f32(N, Nf, bk, Nelements, offset, ggeo, D, lambda, z, p, Ap, partials,
                                               lane_sums, S, s);
    case NBX_BF16:
      return axhelm_pcg_dispatch_bf16(N, Nf, bk, Nelements, offset, ggeo, D, lambda, z, p, Ap,
                                                  partials, lane_sums, S, s);
    default:
      return fail(NBX_ERR_UNSUPPORTED, "axhelm_pcg: precision %d", (int)prec);
  }
}

}  // namespace nbx

using namespace nbx;

extern "C" int nbx_axhelm(int N, int Nfields, int bk, nbx_prec prec, nbx_dlong Nelements,
                          nbx_dlong offset, const nbx_dlong* elementList, const void* ggeo,
                          const void* D, const void* lambda, const void* q, void* Aq, void* stream)
{
  if (Nelements < 0) return fail(NBX_ERR_INVALID, "axhelm: Nelements < 0");
  if (Nelements == 0) return NBX_SUCCESS;
  if (!ggeo || !D || !q || !Aq) return fail(NBX_ERR_INVALID, "axhelm: null array");
  if (!bk && !lambda) return fail(NBX_ERR_INVALID, "axhelm: lambda required when bk == 0");
  const int64_t Np = (int64_t)(N + 1) * (N + 1) * (N + 1);
  if (Nfields > 1 && (int64_t)offset < (int64_t)Nelements * Np && !elementList)
    return fail(NBX_ERR_INVALID, "axhelm: offset %d < Nelements*Np", offset);
  if (!bk && (int64_t)offset < (int64_t)Nelements * Np && !elementList)
    return fail(NBX_ERR_INVALID, "axhelm: lambda offset %d < Nelements*Np", offset);
  return axhelm_launch(N, Nfields, bk, prec, Nelements, offset, elementList, ggeo, D, lambda, q, Aq, nullptr,
                       as_stream(stream));
}

extern "C" int nbx_axhelm_by_name(const char* kernelName, int N, nbx_dlong Nelements, nbx_dlong offset,
                                  const nbx_dlong* elementList, const double* ggeo, const double* D,
                                  const double* lambda, const double* q, double* Aq, void* stream)
{
  if (!kernelName) return fail(NBX_ERR_INVALID, "axhelm_by_name: null name");
  // grammar: axhelm[Partial][_bk][_n3]_v<k>   (nekBone/setup.cpp:313-320)
  const char* p = kernelName;
  if (strncmp(p, "axhelm", 6) != 0) return fail(NBX_ERR_INVALID, "unknown kernel '%s'", kernelName);
  p += 6;
  bool partial = false, bk = false;
  int nf = 1;
  if (strncmp(p, "Partial", 7) == 0) { partial = true; p += 7; }
  if (strncmp(p, "_bk", 3) == 0) { bk = true; p += 3; }
  if (strncmp(p, "_n", 2) == 0) {
    char* end = nullptr;
    nf = (int)strtol(p + 2, &end, 10);
    p = end;
  }
  if (strncmp(p, "_v", 2) != 0) return fail(NBX_ERR_INVALID, "kernel '%s': missing _v<k>", kernelName);
  char* end = nullptr;
  const long ver = strtol(p + 2, &end, 10);
  if (end == p + 2 || *end != '\0' || ver < 0) return fail(NBX_ERR_INVALID, "kernel '%s': bad version", kernelName);
  if (partial && !elementList) return fail(NBX_ERR_INVALID, "kernel '%s' needs an elementList", kernelName);
  if (!partial && elementList) return fail(NBX_ERR_INVALID, "kernel '%s' takes no elementList", kernelName);
  return nbx_axhelm(N, nf, bk ? 1 : 0, NBX_F64, Nelements, offset, elementList, ggeo, D, lambda, q, Aq,
                    stream);
}

extern "C" int nbx_update_jacobi_local(int N, nbx_dlong Nelements, nbx_dlong offset, const int32_t* mapB,
                                       const double* ggeo, const double* D, const double* lambda,
                                       double* diagA, void* stream)
{
  if (Nelements <= 0) return Nelements == 0 ? NBX_SUCCESS : fail(NBX_ERR_INVALID, "jacobi: Nelements < 0");
  if (!ggeo || !D || !lambda || !diagA) return fail(NBX_ERR_INVALID, "jacobi: null array");
  hipStream_t s = as_stream(stream);
  switch (N) {
#define NBX_J_CASE(NV)                                                                              \
  case NV:                                                                                          \
    hipLaunchKernelGGL(k_jacobi<NV + 1>, dim3(Nelements), dim3((NV + 1) * (NV + 1)), 0, s, Nelements, \
                       offset, mapB, ggeo, D, lambda, diagA);                                       \
    NBX_HIP_LAUNCH();                                                                               \
    return NBX_SUCCESS;
    NBX_J_CASE(1)
    NBX_J_CASE(2)
    NBX_J_CASE(3)
    NBX_J_CASE(4)
    NBX_J_CASE(5)
    NBX_J_CASE(6)
    NBX_J_CASE(7)
    NBX_J_CASE(8)
    NBX_J_CASE(9)
    NBX_J_CASE(10)
    NBX_J_CASE(11)
    NBX_J_CASE(12)
    NBX_J_CASE(13)
    NBX_J_CASE(14)
    NBX_J_CASE(15)
#undef NBX_J_CASE
    default:
      return fail(NBX_ERR_UNSUPPORTED, "jacobi: N=%d not supported", N);
  }
}
