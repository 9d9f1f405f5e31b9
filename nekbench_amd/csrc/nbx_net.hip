// Learned element preconditioner: a small 3-D convolutional network over the
// 8x8x8 GLL nodes of one element, inputs the residual and the 7 geometric
// factors, output a correction to Jacobi:
//
//   s      = max_n |r_n|                     (element scale; exact)
//   rh_n   = (float)(r_n / s)                (residual channel)
//   h1     = relu(b1 + Wg . g_n + sum_tap Wr[tap] rh_{n+tap})       32 channels
//   h2     = relu(b2 + W2^T h1)                                        32 channels
//   y_n    = b3 + sum_tap sum_c W3[tap][c] h2_{n+tap}[c]               1 channel
//   z_n    = invDiag_n (r_n + s y_n)          (assembled afterwards by gs)
//
// taps are the 27 neighbours (dz,dy,dx) in {-1,0,1}^3, index
// (dz+1)*9 + (dy+1)*3 + (dx+1), zero padding at the element boundary.  With
// f = 0 the preconditioner is Jacobi exactly.  Weights are bf16 values (held
// in float), arithmetic FP32 with explicit fma, every sum in a fixed order;
// the CPU oracle restates the same order, so forward values and parameter
// gradients are reproduced bit for bit.
//
// One workgroup of 512 lanes per element, lane = node.  The last layer is
// evaluated as T[n][tap] = W3[tap] . h2_n (lane-local) followed by
// y_m = b3 + sum_tap T[m+tap][tap] (27 LDS reads), which keeps LDS traffic at
// 27 values per node.  Weight operands are uniform across the workgroup and
// come through scalar loads.
#include "nbx_internal.h"
#include "nbx_net.h"
#include <cmath>
#include <cstring>
#include <vector>

namespace nbx {

constexpr int kP = 512, kC = 32, kG = 7, kTaps = 27;
constexpr int kPad = 10, kPadN = kPad * kPad * kPad;  // zero-padded tile of the training kernel
constexpr int kFRow = 800;                            // a factor row: node (x, y, z) at 100 z + 10 y + x
// 128 nodes of 96 channel rows; row stride 4 modulo the banks, so the 8 rows
// that 8 lanes read 16 bytes of lie in different banks
constexpr int kTrainRow = 132, kTrainRows = 96;
// T rows in the same buffer: the rows 4 g + u of a product lie 16 banks apart for g = 0..3
constexpr int kTRow = 516;
static_assert(16 * kTRow <= kTrainRows * kTrainRow, "a product's T rows fit the buffer");

typedef float f32x4 __attribute__((ext_vector_type(4)));

// place of the tap's neighbour in the padded tile, relative to the node's 100 z + 10 y + x
__host__ __device__ constexpr int tap_place(int tap)
{
  return 111 + (tap / 9 - 1) * 100 + ((tap / 3) % 3 - 1) * 10 + (tap % 3 - 1);
}

__device__ __forceinline__ int tap_neighbor(int n, int tap)
{
  const int i = n & 7, j = (n >> 3) & 7, k = n >> 6;
  const int dx = tap % 3 - 1, dy = (tap / 3) % 3 - 1, dz = tap / 9 - 1;
  const int ii = i + dx, jj = j + dy, kk = k + dz;
  if ((unsigned)ii > 7u || (unsigned)jj > 7u || (unsigned)kk > 7u) return -1;
  return ii + (jj << 3) + (kk << 6);
}

struct NetFwd {
  float h1[kC];
  float h2[kC];
};

// forward of one node up to T (lane-local); rh in LDS; returns T[27] in T
__device__ __forceinline__ void net_forward_lane(const float* __restrict__ W, int n, const float* s_rh,
                                                 const float (&g)[kG], NetFwd& a, float (&T)[kTaps])
{
  const float* Wr = W + kOffWr;
  const float* Wg = W + kOffWg;
  const float* b1 = W + kOffB1;
  const float* W2 = W + kOffW2;
  const float* b2 = W + kOffB2;
  const float* W3 = W + kOffW3;
#pragma unroll
  for (int c = 0; c < kC; ++c) a.h1[c] = b1[c];
#pragma unroll
  for (int q = 0; q < kG; ++q)
#pragma unroll
    for (int c = 0; c < kC; ++c) a.h1[c] = __builtin_fmaf(Wg[q * kC + c], g[q], a.h1[c]);
#pragma unroll
  for (int tap = 0; tap < kTaps; ++tap) {
    const int nb = tap_neighbor(n, tap);
    if (nb >= 0) {
      const float v = s_rh[nb];
#pragma unroll
      for (int c = 0; c < kC; ++c) a.h1[c] = __builtin_fmaf(Wr[tap * kC + c], v, a.h1[c]);
    }
  }
#pragma unroll
  for (int c = 0; c < kC; ++c) a.h1[c] = a.h1[c] > 0.f ? a.h1[c] : 0.f;
#pragma unroll
  for (int c = 0; c < kC; ++c) a.h2[c] = b2[c];
#pragma unroll
  for (int ci = 0; ci < kC; ++ci)
#pragma unroll
    for (int c = 0; c < kC; ++c) a.h2[c] = __builtin_fmaf(W2[ci * kC + c], a.h1[ci], a.h2[c]);
#pragma unroll
  for (int c = 0; c < kC; ++c) a.h2[c] = a.h2[c] > 0.f ? a.h2[c] : 0.f;
#pragma unroll
  for (int tap = 0; tap < kTaps; ++tap) {
    float t = 0.f;
#pragma unroll
    for (int c = 0; c < kC; ++c) t = __builtin_fmaf(W3[tap * kC + c], a.h2[c], t);
    T[tap] = t;
  }
}

// element scale s = max |r| over the element (block reduction, exact)
__device__ __forceinline__ double element_scale(double rn, double* s_red)
{
  double m = fabs(rn);
#pragma unroll
  for (int h = 32; h >= 1; h >>= 1) m = fmax(m, __shfl_xor(m, h, 64));
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = m;
  __syncthreads();
  double s = s_red[0];
  for (int w = 1; w < kP / 64; ++w) s = fmax(s, s_red[w]);
  return s;
}

// Inference: zl[e*512+n] = w (invDiag (r + s y)), w the assembly weight
// (1/multiplicity, or 1 when w is null); fallback (device flag) turns the
// network off and leaves Jacobi.  Optionally skipped by *skip.
__global__ __launch_bounds__(512) void k_net_apply(const int32_t E, const float* __restrict__ W,
                                                   const float* __restrict__ feat, const double* __restrict__ r,
                                                   const double* __restrict__ invDiag, const double* __restrict__ w,
                                                   double* __restrict__ zl, const int* __restrict__ fallback,
                                                   const int* __restrict__ skip)
{
  if (skip && *skip) return;
  __shared__ float s_rh[kP];
  __shared__ float s_T[kTaps][kP];
  __shared__ double s_red[kP / 64];
  const int n = threadIdx.x;
  const int64_t e = blockIdx.x;
  const int64_t id = e * kP + n;
  const double rn = r[id];
  const double di = invDiag[id];
  const double wn = w ? w[id] : 1.0;
  if (fallback && *fallback) {
    zl[id] = wn * (di * rn);
    return;
  }
  const double s = element_scale(rn, s_red);
  const double inv = s > 0.0 ? 1.0 / s : 0.0;
  s_rh[n] = (float)(rn * inv);
  float g[kG];
#pragma unroll
  for (int q = 0; q < kG; ++q) g[q] = feat[(e * kG + q) * kP + n];
  __syncthreads();
  NetFwd a;
  float T[kTaps];
  net_forward_lane(W, n, s_rh, g, a, T);
#pragma unroll
  for (int tap = 0; tap < kTaps; ++tap) s_T[tap][n] = T[tap];
  __syncthreads();
  float y = W[kOffB3];
#pragma unroll
  for (int tap = 0; tap < kTaps; ++tap) {
    const int nb = tap_neighbor(n, tap);
    if (nb >= 0) y = y + s_T[tap][nb];
  }
  zl[id] = wn * (di * (rn + s * (double)y));
}

// Training: one workgroup per (pair, element) sample, forward and backward;
// the sample's parameter gradient goes to out[sample][kNetPartial], its loss
//   L = inv_norm[pair] sum_n (z_n - e_n)^2
// behind it.  With G non-null the loss is defined outside (energy norm of the
// assembled error) and G[e*512+n] holds its derivative with respect to the
// unweighted element output invDiag (r + s y) at local node n of element e;
// the kernel then back-propagates dL/dy = G invDiag s and reports no loss.
//
// All products run on the matrix cores as 16x16x4 FP32 products, which
// accumulate k in increasing order with one rounding a step: the bits of the
// fma chains they stand for.
// Forward pass and data gradients: a wave takes the 64 nodes of its plane, the
// layers' channels as rows and the nodes as columns; channels are held in the
// order in which one product's result is the next one's operand (NodeChannels).
// The first layer's taps and the last layer's backward taps are read from the
// zero-padded 10^3 tiles of r^ and dL/dy.
// The parameter gradients are products over the 512 nodes, dW[a][c] =
// sum_n A[a][n] B[n][c] in increasing n, one 16x16 tile of one tensor a wave,
// 16 tiles over two phases:
//   phase 1: W3 (taps x channels; dL/dT and h2), W2 (h1 and dL/dpre2)
//   phase 2: Wr, Wg and b1 as 35 rows (r^ taps, factors, ones; dL/dpre1),
//            b2 (ones; dL/dpre2), and b3 as a plain chain beside them.
// The lanes hand their channels to the tiles through LDS 128 nodes at a time,
// nodes ordered inside 16 so that a lane's four k values are one 16-byte
// read; the tap operands are the tiles at a fixed offset, the factors rows of
// the same layout.
// Bound: 4608 products of 32 cycles a sample (123 us of 2048 samples on this
// chip; half of the kernel's time), the rest waits: 80 KB of LDS and 128
// registers keep two workgroups a CU, and a sample has 22 barriers.
// 2048 samples: 3836 us for the form that held one parameter a lane (two LDS
// reads an fma) and gave a workgroup a whole chunk of samples (half the chip
// idle at 16 a chunk); 290 with the forward pass and the data gradients on the
// vector ALUs, lane = node, weights as scalar operands; 248 now.
struct TrainLds {
  float rh[kPadN], dy[kPadN];      // zero-padded tiles
  float g[kG * kFRow];             // factors, node (x, y, z) at 100 z + 10 y + x
  float buf[kTrainRows * kTrainRow];  // T exchange, then 128 nodes of the channels
  double red[kP / 64];
  int nonfinite;                   // dL/dpre1 of some node and channel
};

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The 64 nodes of a wave's plane by 32 channels: node tile tt (nodes 16 tt + col),
// channel tile m; value u is channel 16 m + 4 u + kg.  That is a product's
// result if its rows are the channels in the order of chan_row, and the next
// product's operand at step 4 m + u, whose k = 4 (4 m + u) + kg is the channel:
// the layers chain in registers, each channel's chain in increasing order.
struct NodeChannels {
  f32x4 v[4][2];
};
__device__ __forceinline__ int chan_row(int r) { return 4 * (r & 3) + (r >> 2); }

// acc += A x over STEPS steps of four terms: a(t, m) is the lane's weight of
// channel tile m (those of AHEAD steps in registers at once), x(t, tt) its
// operand of node tile tt
template <int STEPS, int AHEAD, typename WA, typename X>
__device__ __forceinline__ void layer(WA&& a, X&& x, NodeChannels& acc)
{
#pragma unroll
  for (int t0 = 0; t0 < STEPS; t0 += AHEAD) {
    float w[AHEAD][2];
#pragma unroll
    for (int t = t0; t < min(t0 + AHEAD, STEPS); ++t)
#pragma unroll
      for (int m = 0; m < 2; ++m) w[t - t0][m] = a(t, m);
#pragma unroll
    for (int t = t0; t < min(t0 + AHEAD, STEPS); ++t)
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        const float b = x(t, tt);
#pragma unroll
        for (int m = 0; m < 2; ++m) acc.v[tt][m] = mfma4(w[t - t0][m], b, acc.v[tt][m]);
      }
  }
}

template <typename F>
__device__ __forceinline__ void each_channel(F&& f)
{
#pragma unroll
  for (int tt = 0; tt < 4; ++tt)
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int u = 0; u < 4; ++u) f(tt, m, u);
}

// (the values are opaque afterwards: relu' compares them again, or the compiler
// keeps 64 comparisons in scalar registers and spills them)
__device__ __forceinline__ void relu(NodeChannels& h)
{
  each_channel([&](int tt, int m, int u) {
    float v = h.v[tt][m][u] > 0.f ? h.v[tt][m][u] : 0.f;
    asm volatile("" : "+v"(v));
    h.v[tt][m][u] = v;
  });
}

// Rows row .. row + 3 of the first layer's gradient (taps, then factors), one
// channel, over the 128 nodes of the planes k0 and k0 + 1, where some dL/dpre1
// is not finite: a tap whose neighbour lies outside of the element takes no
// part, while the products would multiply its padding, and 0 inf is not 0.
__device__ __forceinline__ void taps_in_range(const TrainLds& lds, const int row, const int channel, const int k0,
                                           f32x4& acc)
{
#pragma unroll 1
  for (int u = 0; u < 4; ++u) {
    const int r = row + u, tap = min(r, kTaps - 1);
    const int dx = r < kTaps ? tap % 3 - 1 : 0, dy = r < kTaps ? (tap / 3) % 3 - 1 : 0, dz = r < kTaps ? tap / 9 - 1 : 0;
    const float* const a = r < kTaps ? lds.rh + tap_place(tap) : lds.g + (r - kTaps) * kFRow;
    float v = u == 0 ? acc[0] : u == 1 ? acc[1] : u == 2 ? acc[2] : acc[3];
#pragma unroll 1
    for (int m = 0; m < 128; ++m) {
      const int i = m & 7, j = (m >> 3) & 7, k = k0 + (m >> 6);
      const bool in = (unsigned)(i + dx) < 8u && (unsigned)(j + dy) < 8u && (unsigned)(k + dz) < 8u;
      const float b = lds.buf[channel * kTrainRow + (m & ~15) + 4 * (m & 3) + ((m & 15) >> 2)];
      if (in) v = __builtin_fmaf(a[100 * k + 10 * j + i], b, v);
    }
    if (u == 0) acc[0] = v;
    else if (u == 1) acc[1] = v;
    else if (u == 2) acc[2] = v;
    else acc[3] = v;
  }
}

__global__ __launch_bounds__(512, 4) void k_net_train(const int2* __restrict__ samples, const int64_t pairStride,
                                                      const float* __restrict__ R, const float* __restrict__ Ev,
                                                      const double* __restrict__ invNorm, const float* __restrict__ W,
                                                      const float* __restrict__ feat,
                                                      const double* __restrict__ invDiag,
                                                      const double* __restrict__ G, float* __restrict__ out)
{
  __shared__ TrainLds lds;
  const int n = threadIdx.x, l = n & 63, wv = n >> 6, col = l & 15, kg = l >> 4;
  const int i = n & 7, j = (n >> 3) & 7, k = n >> 6;
  const int place = 100 * k + 10 * j + i;  // in the 10-strided layout; the tiles' interior starts at 111
  const float* W2 = W + kOffW2;
  const float* W3 = W + kOffW3;
  const int2 pe = samples[blockIdx.x];
  const int64_t e = pe.y;
  const int64_t off = (int64_t)pe.x * pairStride + e * kP + n;
  const double rn = (double)R[off];
  const double en = G ? 0.0 : (double)Ev[off];
  const double di = invDiag[e * kP + n];
  for (int q = n; q < kPadN; q += kP) lds.rh[q] = lds.dy[q] = 0.f;
  if (n == 0) lds.nonfinite = 0;
#pragma unroll
  for (int q = 0; q < kG; ++q) lds.g[q * kFRow + place] = feat[(e * kG + q) * kP + n];
  const double s = element_scale(rn, lds.red);  // its barrier also ends the zero fill
  const double inv = s > 0.0 ? 1.0 / s : 0.0;
  lds.rh[111 + place] = (float)(rn * inv);
  __syncthreads();
  // the lane's nodes in the products are those of its wave's plane, tile tt's
  // at pl + 20 tt; its weights' rows are channels 16 m + ch
  const int pl = 100 * wv + 10 * (col >> 3) + (col & 7), ch = chan_row(col);
  const float* const lds0 = reinterpret_cast<const float*>(&lds);  // rh, dy, g in that order
  NodeChannels h1, h2;
  each_channel([&](int tt, int m, int u) { h1.v[tt][m][u] = W[kOffB1 + 16 * m + 4 * u + kg]; });
  {
    // terms: the factors, then the taps (zero past the last)
    constexpr int kTerms = kG + kTaps, kSteps = (kTerms + 3) / 4;
    int at[kSteps], wt[kSteps];
#pragma unroll
    for (int t = 0; t < kSteps; ++t) {
      const int term = 4 * t + kg, tap = min(max(term - kG, 0), kTaps - 1);
      at[t] = pl + (term < kG ? 2 * kPadN + term * kFRow : tap_place(tap));
      wt[t] = (term < kG ? kOffWg + term * kC : kOffWr + tap * kC) + ch;
    }
    layer<kSteps, kSteps>([&](int t, int m) { return 4 * t + kg < kTerms ? W[wt[t] + 16 * m] : 0.f; },
                  [&](int t, int tt) {
                    const float v = lds0[at[t] + 20 * tt];
                    return 4 * t + 3 < kTerms || 4 * t + kg < kTerms ? v : 0.f;
                  },
                  h1);
  }
  relu(h1);
  each_channel([&](int tt, int m, int u) { h2.v[tt][m][u] = W[kOffB2 + 16 * m + 4 * u + kg]; });
  layer<kC / 4, 8>([&](int t, int m) { return W2[(4 * t + kg) * kC + 16 * m + ch]; },
                [&](int t, int tt) { return h1.v[tt][t >> 2][t & 3]; }, h2);
  relu(h2);
  // y = b3 + sum over the taps of T[tap] at node n + tap: a product's 16 taps at
  // a time through the buffer
  const bool ox[3] = {i > 0, true, i < 7}, oy[3] = {j > 0, true, j < 7}, oz[3] = {k > 0, true, k < 7};
  float y = W[kOffB3];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    f32x4 T[4] = {};
    float w[kC / 4];
#pragma unroll
    for (int t = 0; t < kC / 4; ++t) w[t] = W3[min(16 * m + col, kTaps - 1) * kC + 4 * t + kg];
#pragma unroll
    for (int t = 0; t < kC / 4; ++t)
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) T[tt] = mfma4(w[t], h2.v[tt][t >> 2][t & 3], T[tt]);
    if (m) __syncthreads();  // the first taps' readers are done
#pragma unroll
    for (int tt = 0; tt < 4; ++tt)
#pragma unroll
      for (int u = 0; u < 4; ++u) lds.buf[(4 * kg + u) * kTRow + 64 * wv + 16 * tt + col] = T[tt][u];
    __syncthreads();
#pragma unroll
    for (int tap = 16 * m; tap < min(16 * m + 16, kTaps); ++tap) {
      const int dx = tap % 3, dyy = (tap / 3) % 3, z = tap / 9;
      const bool in = ox[dx] && oy[dyy] && oz[z];
      const int nb = n + (dx - 1) + 8 * (dyy - 1) + 64 * (z - 1);
      const float v = lds.buf[(tap - 16 * m) * kTRow + (in ? nb : n)];
      y = y + (in ? v : 0.f);
    }
  }
  const double zz = di * (rn + s * (double)y);
  const double res = zz - en;
  const double wn = G ? 0.0 : invNorm[pe.x];
  const float dy = G ? (float)(G[e * kP + n] * di * s) : (float)(2.0 * res * wn * di * s);
  lds.dy[111 + place] = dy;
  // loss: lane values, fixed tree (per-wave halving, waves in order)
  if (!G) {
    double v = res * res * wn;
#pragma unroll
    for (int h = 32; h >= 1; h >>= 1) v += __shfl_xor(v, h, 64);
    if (l == 0) lds.red[wv] = v;
  }
  __syncthreads();
  float* const po = out + (int64_t)blockIdx.x * kNetPartial;
  if (n == 0) {
    double t = 0.0;
    if (!G) {
      t = lds.red[0];
      for (int w = 1; w < kP / 64; ++w) t = t + lds.red[w];
    }
    reinterpret_cast<double*>(po + kNetParamsPadded)[0] = t;
  }
  // dL/dpre2 = relu'(h2) sum over the taps of W3[tap] dy(n - tap)
  NodeChannels d2 = {};
  {
    constexpr int kSteps = (kTaps + 3) / 4;
    int at[kSteps];
#pragma unroll
    for (int t = 0; t < kSteps; ++t) at[t] = kPadN + pl + tap_place(26 - min(4 * t + kg, kTaps - 1));
    layer<kSteps, 4>([&](int t, int m) { return 4 * t + kg < kTaps ? W3[(4 * t + kg) * kC + 16 * m + ch] : 0.f; },
                  [&](int t, int tt) {
                    const float v = lds0[at[t] + 20 * tt];
                    return 4 * t + 3 < kTaps || 4 * t + kg < kTaps ? v : 0.f;
                  },
                  d2);
  }
  each_channel([&](int tt, int m, int u) { d2.v[tt][m][u] = h2.v[tt][m][u] > 0.f ? d2.v[tt][m][u] : 0.f; });

  // the node's column in a 128-node buffer row: inside 16 nodes, 4 s + g is
  // kept at 4 g + s, so k group g reads the nodes 4 s + g, s = 0..3, at once
  const int cpos = (wv & 1) * 64 + ((col & 3) << 2) + (col >> 2);
  auto put = [&](int row0, const NodeChannels& x) {
    each_channel([&](int tt, int m, int u) {
      lds.buf[(row0 + 16 * m + 4 * u + kg) * kTrainRow + cpos + 16 * tt] = x.v[tt][m][u];
    });
  };
  const int rd = col * kTrainRow + 4 * kg;  // a lane's operand read: row col, group kg
  // phase 1: waves 0..3 W3, waves 4..7 W2; one (row tile, channel tile) each
  {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    const int rt = (wv >> 1) & 1, ct = wv & 1;
    const int tap = min(16 * rt + col, kTaps - 1);  // rows past the taps are not stored
    const float* const ay = lds.dy + tap_place(26 - tap) + kg;
    for (int h = 0; h < 4; ++h) {
      __syncthreads();  // the buffer's last readers are done
      if ((wv >> 1) == h) {
        put(0, h2);
        put(kC, h1);
        put(2 * kC, d2);
      }
      __syncthreads();
      if (wv < 4) {
        const float* const b = lds.buf + 16 * ct * kTrainRow + rd;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const f32x4 bv = *reinterpret_cast<const f32x4*>(b + 16 * q);
#pragma unroll
          for (int u = 0; u < 4; ++u)
            acc = mfma4(ay[200 * h + 100 * (q / 4) + 10 * ((2 * q + u / 2) % 8) + 4 * (u % 2)], bv[u], acc);
        }
      } else {
        const float* const a = lds.buf + (kC + 16 * rt) * kTrainRow + rd;
        const float* const b = lds.buf + (2 * kC + 16 * ct) * kTrainRow + rd;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const f32x4 av = *reinterpret_cast<const f32x4*>(a + 16 * q), bv = *reinterpret_cast<const f32x4*>(b + 16 * q);
#pragma unroll
          for (int u = 0; u < 4; ++u) acc = mfma4(av[u], bv[u], acc);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int row = 16 * rt + 4 * kg + u;
      if (wv >= 4) po[kOffW2 + row * kC + 16 * ct + col] = acc[u];
      else if (row < kTaps) po[kOffW3 + row * kC + 16 * ct + col] = acc[u];
    }
  }
  // dL/dpre1 = relu'(h1) W2 dL/dpre2
  NodeChannels d1 = {};
  layer<kC / 4, 8>([&](int t, int m) { return W2[(16 * m + ch) * kC + 4 * t + kg]; },
                [&](int t, int tt) { return d2.v[tt][t >> 2][t & 3]; }, d1);
  each_channel([&](int tt, int m, int u) { d1.v[tt][m][u] = h1.v[tt][m][u] > 0.f ? d1.v[tt][m][u] : 0.f; });
  {
    float z[4] = {};  // not zero where a value is not finite
    each_channel([&](int tt, int m, int u) { z[tt] = __builtin_fmaf(d1.v[tt][m][u], 0.f, z[tt]); });
    const float zero = (z[0] + z[1]) + (z[2] + z[3]);
    if (!(zero == 0.f)) lds.nonfinite = 1;
  }
  // phase 2: waves 0..5 the 35 rows of Wr, Wg, b1 (three row tiles), waves 6, 7 b2
  {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    const int rt = wv >> 1, ct = wv & 1;
    const int row0 = 16 * rt + col;  // this lane's A row
    const bool one = rt == 3 || row0 >= kTaps + kG;
    const float* const ax =
        (row0 < kTaps ? lds.rh + tap_place(row0) : lds.g + (one ? 0 : row0 - kTaps) * kFRow) + kg;
    float b3 = 0.f;
    for (int h = 0; h < 4; ++h) {
      __syncthreads();
      if ((wv >> 1) == h) {
        put(0, d1);
        put(kC, d2);
      }
      __syncthreads();
      if (rt < 2 && lds.nonfinite) {
        taps_in_range(lds, 16 * rt + 4 * kg, 16 * ct + col, 2 * h, acc);
        continue;
      }
      const float* const b = lds.buf + ((rt == 3 ? kC : 0) + 16 * ct) * kTrainRow + rd;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const f32x4 bv = *reinterpret_cast<const f32x4*>(b + 16 * q);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int at = 200 * h + 100 * (q / 4) + 10 * ((2 * q + u / 2) % 8) + 4 * (u % 2);
          const float a = one ? 1.f : ax[at];
          acc = mfma4(a, bv[u], acc);
          if (wv == 7) {  // b3: nodes in order, beside the products
            const float* const d = lds.dy + 111 + at;
#pragma unroll
            for (int x = 0; x < 4; ++x) b3 = b3 + d[x];
          }
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int row = 16 * rt + 4 * kg + u;
      if (rt == 3) {
        if (row == 48) po[kOffB2 + 16 * ct + col] = acc[u];
      } else if (row < kTaps) {
        po[kOffWr + row * kC + 16 * ct + col] = acc[u];
      } else if (row < kTaps + kG) {
        po[kOffWg + (row - kTaps) * kC + 16 * ct + col] = acc[u];
      } else if (row == kTaps + kG) {
        po[kOffB1 + 16 * ct + col] = acc[u];
      }
    }
    if (n == kP - 1) po[kOffB3] = b3;
  }
}

// partials[b][q]: the sum over chunk b's samples, in order, of the sample
// gradients (and losses); the samples of this launch are first .. first +
// count - 1 of the batch, and a chunk begun in an earlier launch goes on from
// its partial.
__global__ __launch_bounds__(256) void k_net_chunk_sum(const int32_t first, const int32_t count, const int32_t chunk,
                                                       const float* __restrict__ grads, float* __restrict__ partials)
{
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  const int32_t b = first / chunk + (int32_t)blockIdx.y;
  const int32_t s0 = max(first, (int32_t)((int64_t)b * chunk));
  const int32_t s1 = (int32_t)min((int64_t)first + count, (int64_t)(b + 1) * chunk);
  const bool goes_on = s0 != (int64_t)b * chunk;
  float* const pb = partials + (int64_t)b * kNetPartial;
  const float* const g = grads + (int64_t)(s0 - first) * kNetPartial;
  if (q < kNetParams) {
    float acc = goes_on ? pb[q] : 0.f;
#pragma unroll 8
    for (int32_t i = 0; i < s1 - s0; ++i) acc = acc + g[(int64_t)i * kNetPartial + q];
    pb[q] = acc;
  } else if (q == kNetParamsPadded) {
    double acc = goes_on ? reinterpret_cast<const double*>(pb + kNetParamsPadded)[0] : 0.0;
#pragma unroll 8
    for (int32_t i = 0; i < s1 - s0; ++i)
      acc = acc + reinterpret_cast<const double*>(g + (int64_t)i * kNetPartial + kNetParamsPadded)[0];
    reinterpret_cast<double*>(pb + kNetParamsPadded)[0] = acc;
  }
}

// grad[q] = sum over chunks (in order) of partials[b][q]; loss likewise
// (a serial chain of loads: 32 in flight, 44 -> 12 us for 128 chunks)
__global__ __launch_bounds__(64) void k_net_grad_sum(const int32_t nblocks, const float* __restrict__ partials,
                                                     float* __restrict__ grad, double* __restrict__ loss)
{
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < kNetParams) {
    float acc = 0.f;
    int b = 0;
    for (; b + 32 <= nblocks; b += 32) {
      float t[32];
#pragma unroll
      for (int u = 0; u < 32; ++u) t[u] = partials[(int64_t)(b + u) * kNetPartial + q];
#pragma unroll
      for (int u = 0; u < 32; ++u) acc = acc + t[u];
    }
    for (; b < nblocks; ++b) acc = acc + partials[(int64_t)b * kNetPartial + q];
    grad[q] = acc;
  } else if (q == kNetParams) {
    double acc = 0.0;
#pragma unroll 16
    for (int b = 0; b < nblocks; ++b)
      acc = acc + reinterpret_cast<const double*>(partials + (int64_t)b * kNetPartial + kNetParamsPadded)[0];
    *loss = acc;
  }
}

__device__ __forceinline__ float round_bf16(float x) { return bf16_round(x); }

// Adam on FP32 master weights; the forward weights are their bf16 rounding
__global__ __launch_bounds__(256) void k_net_adam(const int32_t np, float* __restrict__ master,
                                                  float* __restrict__ m, float* __restrict__ v,
                                                  const float* __restrict__ grad, float* __restrict__ wbf,
                                                  const float lr, const float b1, const float b2, const float eps,
                                                  const float c1, const float c2)
{
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= np) return;
  const float g = grad[q];
  const float mq = b1 * m[q] + (1.f - b1) * g;
  const float vq = b2 * v[q] + (1.f - b2) * g * g;
  m[q] = mq;
  v[q] = vq;
  const float upd = lr * (mq / c1) / (sqrtf(vq / c2) + eps);
  const float w = master[q] - upd;
  master[q] = w;
  wbf[q] = round_bf16(w);
}

// normalised geometric features: feat[e][q][n] = ggeo[e][q][n] / scale[q]
__global__ __launch_bounds__(256) void k_net_features(const int64_t n, const double* __restrict__ ggeo,
                                                      const double* __restrict__ invScale, float* __restrict__ feat)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int q = (int)((i / kP) % kG);
  feat[i] = (float)(ggeo[i] * invScale[q]);
}

int net_apply_launch(int32_t E, const float* W, const float* feat, const double* r, const double* invDiag,
                     const double* w, double* zl, const int* fallback, const int* skip, hipStream_t s)
{
  hipLaunchKernelGGL(k_net_apply, dim3(E), dim3(kP), 0, s, E, W, feat, r, invDiag, w, zl, fallback, skip);
  NBX_HIP_LAUNCH();
  return NBX_SUCCESS;
}

// samples first .. first + count - 1 of a batch: their gradients into grads
// (count rows of kNetPartial), summed into the chunks' partials
int net_train_launch(int32_t first, int32_t count, int32_t chunk, const int2* samples, int64_t pairStride,
                     const float* R, const float* Ev, const double* invNorm, const float* W, const float* feat,
                     const double* invDiag, const double* G, float* grads, float* partials, hipStream_t s)
{
  hipLaunchKernelGGL(k_net_train, dim3(count), dim3(kP), 0, s, samples + first, pairStride, R, Ev, invNorm, W, feat,
                     invDiag, G, grads);
  NBX_HIP_LAUNCH();
  const int32_t chunks = (first + count - 1) / chunk - first / chunk + 1;
  hipLaunchKernelGGL(k_net_chunk_sum, dim3((kNetPartial + 255) / 256, chunks), dim3(256), 0, s, first, count, chunk,
                     grads, partials);
  NBX_HIP_LAUNCH();
  return NBX_SUCCESS;
}

int net_grad_sum_launch(int32_t nblocks, const float* partials, float* grad, double* loss, hipStream_t s)
{
  hipLaunchKernelGGL(k_net_grad_sum, dim3((kNetParams + 1 + 63) / 64), dim3(64), 0, s, nblocks, partials, grad, loss);
  NBX_HIP_LAUNCH();
  return NBX_SUCCESS;
}

int net_adam_launch(float* master, float* m, float* v, const float* grad, float* wbf, float lr, int step,
                    hipStream_t s)
{
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(k_net_adam, dim3((kNetParams + 255) / 256), dim3(256), 0, s, kNetParams, master, m, v, grad, wbf,
                     lr, b1, b2, eps, c1, c2);
  NBX_HIP_LAUNCH();
  return NBX_SUCCESS;
}

int net_features_launch(int32_t E, const double* ggeo, const double* invScale, float* feat, hipStream_t s)
{
  const int64_t n = (int64_t)E * kG * kP;
  hipLaunchKernelGGL(k_net_features, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, ggeo, invScale, feat);
  NBX_HIP_LAUNCH();
  return NBX_SUCCESS;
}

}  // namespace nbx
