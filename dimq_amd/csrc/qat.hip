// Training-side DIMQ kernels (the QAT step before the packed path):
//  * the Gibbs softmin distortion  L = sum_i -tau (logsumexp_j(-d_ij / tau) - log K),
//    d_ij = (w_i - c_j)^2  (dimq_softmin_loss, quant/dimq.py:244-273), forward and
//    backward;
//  * soft dequantization  out_i = sum_j p_ij c_j,  p_ij = softmax_j(-d_ij / tau)
//    (soft_dequantize_weight, quant/dimq.py:224-241), forward and backward;
//  * the hinge separation loss over centre pairs with margin
//    delta = eta * 6 * std(w) / K  (separation_loss, quant/dimq.py:276-296) and
//    its gradient in the centres.
// Everything is computed in fp32 from w.float() and centres.float(), as the
// reference does.  The centres (K <= 256) sit in LDS.  Exponents are formed as
// -(d_ij - dmin_i) / tau with dmin_i = min_j d_ij (exact 0 at the nearest
// centre, no cancellation of two large terms at small tau), so
//   logsumexp_j(-d_ij / tau) = -dmin_i / tau + log s_i,
//   s_i = sum_j exp(-(d_ij - dmin_i) / tau),   p_ij = exp(-(d_ij - dmin_i) / tau) / s_i,
// and the softmin term is dmin_i - tau log(s_i / K).  For s_i > K / 2
// (near-uniform p: large tau) log(s_i / K) is formed as
// log1p(sum_j expm1(-(d_ij - dmin_i) / tau) / K), since log s_i - log K would
// cancel to a few digits there; otherwise as log s_i - log K.  The forward
// kernels store (dmin_i, 1 / s_i) per element, so a backward pass gets p_ij
// without a second pass over the centres (and with no rounding of a logarithm in
// its exponent).  Sums over elements (the loss, the centre gradients) go through
// per-work-group partials and a final pass in a fixed order: results do not
// depend on scheduling.
#include <type_traits>

#include "common.h"

namespace dimq {
namespace {

constexpr int kQatThreads = 256;
constexpr int kQatEpt = 4;                         // elements per thread and trip
constexpr int kQatChunk = kQatThreads * kQatEpt;  // elements per work-group and trip
constexpr int kQatTile = 16;                       // centres per gradient tile
// Above this many chunks a work-group takes several (all about equally many):
// it keeps its sums over all of them, so the final pass has at most this many
// rows to add whatever n is.
constexpr int64_t kQatMaxBlocks = 8192;

constexpr double kLog2e = 1.4426950408889634074;

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  return v;
}

__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int wave = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// Sums of 16 per-lane values over the wave: after each of four exchange steps
// a lane holds half as many values of twice as many lanes (15 exchanges
// instead of the 96 of 16 separate butterflies), then two plain steps.  Lane
// l's result is the sum of value (l >> 2) & 15 in bit-reversed order of the
// exchanges: 8 (l bit 5), 4 (bit 4), 2 (bit 3), 1 (bit 2).
__device__ __forceinline__ float wave_sum16(float (&v)[16]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int h = 8; h >= 1; h >>= 1) {
    const bool up = (lane & (4 * h)) != 0;
#pragma unroll
    for (int i = 0; i < h; ++i) {
      const float lo = v[i], hi = v[i + h];  // values, not places: a place chosen at run time moves v to LDS
      v[i] = (up ? hi : lo) + __shfl_xor(up ? lo : hi, 4 * h, 64);
    }
  }
  float r = v[0];
  r += __shfl_xor(r, 2, 64);
  r += __shfl_xor(r, 1, 64);
  return r;  // of value index (lane >> 2) & 15
}

// (w - c)^2 rounded to fp32 once, as the reference's (w - c).pow(2): never
// contracted into a later subtraction (hipcc contracts a * b - c into an fma
// by default; an exact square there differs from dmin's rounded one, and at
// small tau that difference times 1/tau moves the exponent by O(1))
__device__ __forceinline__ float sqd(float w, float c) {
#pragma clang fp contract(off)
  const float d = w - c;
  return d * d;
}

// exp(-(d2 - dmin) / tau) with il = log2(e) / tau rounded once from double:
// one product and the hardware's base-2 exponential (1 ulp) in place of a
// product, a range reduction and the library's expf; the exponent's relative
// error is the same two roundings.  Exponents are clamped at 2^-150: such a
// term cannot change a sum that holds exp(0) = 1.
__device__ __forceinline__ float pexp(float d2, float dmin, float il) {
#pragma clang fp contract(off)
  return __builtin_amdgcn_exp2f(fmaxf((dmin - d2) * il, -150.0f));
}

// exp(x) - 1 for x = -(d2 - dmin) / tau <= 0, small x kept exactly: its series
// to x^9 / 9! down to -0.5 (relative truncation below 1e-8), the exponential
// itself minus 1 further down, where nothing cancels.
__device__ __forceinline__ float pexpm1(float d2, float dmin, float inv_tau, float il) {
  const float x = fmaxf(-(d2 - dmin) * inv_tau, -100.0f);
  float t = fmaf(x, 1.0f / 9.0f, 1.0f);
  t = fmaf(x * (1.0f / 8.0f), t, 1.0f);
  t = fmaf(x * (1.0f / 7.0f), t, 1.0f);
  t = fmaf(x * (1.0f / 6.0f), t, 1.0f);
  t = fmaf(x * (1.0f / 5.0f), t, 1.0f);
  t = fmaf(x * (1.0f / 4.0f), t, 1.0f);
  t = fmaf(x * (1.0f / 3.0f), t, 1.0f);
  t = fmaf(x * (1.0f / 2.0f), t, 1.0f);
  return x > -0.5f ? x * t : pexp(d2, dmin, il) - 1.0f;
}

// The thread's elements of a chunk; the dtype is switched on once, so
// the loads go out together.  Elements past the end re-load the last one.
template <int E>
__device__ __forceinline__ void load_ept(const void* p, int dt, const int64_t (&at)[E], float (&v)[E]) {
  switch (dt) {
    case DIMQ_F32:
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = reinterpret_cast<const float*>(p)[at[e]];
      return;
    case DIMQ_F16:
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = f16_bits_to_float(reinterpret_cast<const uint16_t*>(p)[at[e]]);
      return;
    case DIMQ_BF16:
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = bf16_bits_to_float(reinterpret_cast<const uint16_t*>(p)[at[e]]);
      return;
    default:
#pragma unroll
      for (int e = 0; e < E; ++e) v[e] = (float)reinterpret_cast<const double*>(p)[at[e]];
  }
}

// The centres of a kernel instance.  KT = 4, 8, 16: exactly that many (the
// codebooks of 2, 3 and 4 bits), in scalar registers, every loop over them
// unrolled with no branch, so that the elements' chains interleave over all
// centres (a test per centre ends a basic block at each: softmin forward at
// 16 centres 20.1 us with it, 18.1 without).  KT = kAnyTo16: any K up to 16
// the same way, with that test.  KT = 0: any K <= 256 from LDS (one broadcast
// read serves a thread's four elements).
constexpr int kAnyTo16 = 17;
constexpr int centre_regs(int kt) { return kt == kAnyTo16 ? 16 : kt > 0 ? kt : 1; }

template <int KT>
struct Centres {
  float c[centre_regs(KT)];
  const float* cs;
  int K;
  __device__ __forceinline__ void load(const float* __restrict__ g, int K_, float* lds) {
    K = K_;
    cs = lds;
    if (KT > 0) {
#pragma unroll
      for (int j = 0; j < centre_regs(KT); ++j) c[j] = g[KT != kAnyTo16 || j < K ? j : K - 1];
    } else {
      for (int j = threadIdx.x; j < K; j += kQatThreads) lds[j] = g[j];
      __syncthreads();
    }
  }
  // f(j, centre j) over the K centres in order
  template <class F>
  __device__ __forceinline__ void each(F f) const {
    if (KT > 0) {
#pragma unroll
      for (int j = 0; j < centre_regs(KT); ++j)
        if (KT != kAnyTo16 || j < K) f(j, c[j]);
    } else {
#pragma unroll 4
      for (int j = 0; j < K; ++j) f(j, cs[j]);
    }
  }
};

// MODE 0: softmin loss partials (+ aux);  MODE 1: soft dequantization (+ aux).
// VALU-bound: per element and centre a distance and a minimum, then the
// distance again, one hardware exponential and one or two sums (out is
// sum e_j c_j / sum e_j in the same pass).  2,359,296 fp32 weights, 16
// centres: softmin with its final pass 17.8 us (25.3 us before that pass with
// expf), soft dequantization 42.9 -> 15.0 us.
template <int MODE, int KT>
__global__ __launch_bounds__(kQatThreads) void qat_forward_kernel(const void* __restrict__ w, int wdt, int64_t n,
                                                                  const float* __restrict__ c, int K, float inv_tau,
                                                                  float il, float tau, float2* __restrict__ aux,
                                                                  float* __restrict__ partial, void* __restrict__ out) {
  __shared__ float cs[KT > 0 ? 1 : 256];
  __shared__ float red[4];
  Centres<KT> ct;
  ct.load(c, K, cs);
  const float fK = static_cast<float>(K);
  const float logK = logf(fK);
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kQatChunk;
  float acc = 0.0f;
  for (int64_t base = static_cast<int64_t>(blockIdx.x) * kQatChunk; base < n; base += stride) {
    int64_t at[kQatEpt];
    float wv[kQatEpt], dmin[kQatEpt], s4[4][kQatEpt], o[kQatEpt];
#pragma unroll
    for (int e = 0; e < kQatEpt; ++e) {
      const int64_t i = base + e * kQatThreads + threadIdx.x;
      at[e] = i < n ? i : n - 1;
      dmin[e] = __builtin_inff();
      o[e] = s4[0][e] = s4[1][e] = s4[2][e] = s4[3][e] = 0.0f;
    }
    load_ept(w, wdt, at, wv);
    ct.each([&](int, float cj) {
#pragma unroll
      for (int e = 0; e < kQatEpt; ++e) dmin[e] = fminf(dmin[e], fabsf(wv[e] - cj));
    });
    // rounding is monotone: the square of the smallest distance is the smallest rounded square
#pragma unroll
    for (int e = 0; e < kQatEpt; ++e) dmin[e] = dmin[e] * dmin[e];
    // s = sum_j exp(x_j), x_j = -(d_j - dmin) / tau <= 0: in [1, K]; four partial sums keep its rounding small
    ct.each([&](int j, float cj) {
#pragma unroll
      for (int e = 0; e < kQatEpt; ++e) {
        const float p = pexp(sqd(wv[e], cj), dmin[e], il);
        if (KT > 0) {
          s4[j & 3][e] += p;
        } else {  // rotated: the loop's index is no constant
          const float t = s4[0][e] + p;
          s4[0][e] = s4[1][e], s4[1][e] = s4[2][e], s4[2][e] = s4[3][e], s4[3][e] = t;
        }
        if (MODE == 1) o[e] = fmaf(p, cj, o[e]);
      }
    });
#pragma unroll
    for (int e = 0; e < kQatEpt; ++e) {
      const float s = (s4[0][e] + s4[1][e]) + (s4[2][e] + s4[3][e]);
      float lsk = 0.0f;
      if (MODE == 0) {
        lsk = logf(s) - logK;
        if (s > 0.5f * fK) {  // near-uniform p: sum_j (exp(x_j) - 1), small terms kept exactly
          float q = 0.0f;
          ct.each([&](int, float cj) { q += pexpm1(sqd(wv[e], cj), dmin[e], inv_tau, il); });
          lsk = log1pf(q / fK);
        }
      }
      if (base + e * kQatThreads + threadIdx.x < n) {
        const float inv = 1.0f / s;  // exactly 1 for a single nearest centre: p is then 1 and out that centre
        if (aux) aux[at[e]] = make_float2(dmin[e], inv);
        if (MODE == 0) {
          acc += dmin[e] - tau * lsk;
        } else {
          store_from_float(out, wdt, at[e], o[e] * inv);
        }
      }
    }
  }
  if (MODE == 0) {
    const float t = block_sum(acc, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = t;
  }
}

// Backward of both forwards:
//   MODE 0 (softmin, upstream scalar g):
//     dL/dw_i = g sum_j p_ij 2 (w_i - c_j),   dL/dc_j = -2 g sum_i p_ij (w_i - c_j)
//   MODE 1 (soft dequantization, upstream g_i, out_i = sum_j p_ij c_j):
//     dL/dw_i = g_i sum_j p_ij (c_j - out_i) (-2 (w_i - c_j) / tau)
//     dL/dc_j = sum_i g_i p_ij (1 + (c_j - out_i) 2 (w_i - c_j) / tau)
// K <= 16: each p_ij is formed once and kept in registers, and the centre sums
// stay in registers over all the work-group's trips (one reduction at its
// end); four work-groups per CU take the trips in turn, two elements per
// thread and trip, the next trip's loads in flight behind this one's
// arithmetic.  Larger K: four elements per thread,
// 16 centres at a time, the tile's sums reduced over the wave and kept in LDS.
// 2,359,296 fp32 weights, 16 centres, with the final pass over the partial
// rows: softmin 19.4 us, soft dequantization 24.0 us (29.5 and 55.7 us before
// that pass when every p was formed with expf and the centre sums were reduced
// by 16 separate butterflies per 1,024 elements).
constexpr int bwd_ept(int kt) { return kt > 0 ? 2 : kQatEpt; }

template <int MODE, int KT>
__global__ __launch_bounds__(kQatThreads) void qat_backward_kernel(const void* __restrict__ w, int wdt, int64_t n,
                                                                   const float* __restrict__ c, int K, float inv_tau,
                                                                   float il, const float2* __restrict__ aux,
                                                                   const float* __restrict__ gscalar,
                                                                   const void* __restrict__ gout, int gdt,
                                                                   void* __restrict__ grad_w, int gwdt,
                                                                   float* __restrict__ partial) {
  constexpr int KR = centre_regs(KT), E = bwd_ept(KT);
  constexpr int64_t kChunk = kQatThreads * E;
  __shared__ float cs[KT > 0 ? 1 : 256];
  __shared__ float red[4][KT > 0 ? kQatTile : 256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kChunk;
  int64_t base = static_cast<int64_t>(blockIdx.x) * kChunk;
  float wn[E], gn[E];
  float2 an[E];
  // a trip's loads; elements past the end re-load the last one
  auto load = [&](int64_t b) {
    int64_t at[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int64_t i = b + e * kQatThreads + threadIdx.x;
      at[e] = i < n ? i : n - 1;
    }
    load_ept(w, wdt, at, wn);
#pragma unroll
    for (int e = 0; e < E; ++e) an[e] = aux[at[e]];
    if (MODE == 1) load_ept(gout, gdt, at, gn);
  };
  load(base);
  Centres<KT> ct;
  ct.load(c, K, cs);
  const float g0 = MODE == 0 ? *gscalar : 0.0f;
  const float two_tau = 2.0f * inv_tau;
  float sums[kQatTile];  // of the registers' centres, over all trips (KT > 0) or of one tile
#pragma unroll
  for (int u = 0; u < kQatTile; ++u) sums[u] = 0.0f;
  if (KT == 0)
    for (int j = lane; j < 256; j += 64) red[wave][j] = 0.0f;  // each wave's own row

  for (; base < n; base += stride) {
    float wv[E], gv[E], ov[E], gw[E], dmin[E], inv[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const bool ok = base + e * kQatThreads + threadIdx.x < n;
      wv[e] = wn[e];
      dmin[e] = an[e].x;
      inv[e] = ok ? an[e].y : 0.0f;  // p = 0 for elements past the end
      gv[e] = MODE == 1 ? gn[e] : g0;
      gw[e] = ov[e] = 0.0f;
    }
    if (base + stride < n) load(base + stride);
    if (KT > 0) {
      float p[KR][E];
      ct.each([&](int j, float cj) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const float pij = pexp(sqd(wv[e], cj), dmin[e], il) * inv[e];
          if (MODE == 0) {
            const float pd = pij * (wv[e] - cj);
            gw[e] += pd;
            sums[j] += pd;
          } else {
            p[j][e] = pij;
            ov[e] = fmaf(pij, cj, ov[e]);
          }
        }
      });
      if (MODE == 1) {
        ct.each([&](int j, float cj) {
#pragma unroll
          for (int e = 0; e < E; ++e) {
            const float q = gv[e] * p[j][e];
            const float t = (cj - ov[e]) * (two_tau * (wv[e] - cj));
            gw[e] -= q * t;
            sums[j] += fmaf(q, t, q);
          }
        });
      }
    } else {
      if (MODE == 1)  // out_i again (the forward's value before its rounding to w's dtype)
        ct.each([&](int, float cj) {
#pragma unroll
          for (int e = 0; e < E; ++e) ov[e] = fmaf(pexp(sqd(wv[e], cj), dmin[e], il) * inv[e], cj, ov[e]);
        });
      for (int t0 = 0; t0 < K; t0 += kQatTile) {
#pragma unroll
        for (int u = 0; u < kQatTile; ++u) {
          float gc = 0.0f;
          if (t0 + u < K) {
            const float cj = cs[t0 + u];
#pragma unroll
            for (int e = 0; e < E; ++e) {
              const float pij = pexp(sqd(wv[e], cj), dmin[e], il) * inv[e];
              if (MODE == 0) {
                const float pd = pij * (wv[e] - cj);
                gw[e] += pd;
                gc += pd;
              } else {
                const float q = gv[e] * pij;
                const float t = (cj - ov[e]) * (two_tau * (wv[e] - cj));
                gw[e] -= q * t;
                gc += fmaf(q, t, q);
              }
            }
          }
          sums[u] = gc;
        }
        const float r = wave_sum16(sums);
        if ((lane & 3) == 0) red[wave][t0 + (lane >> 2)] += r;  // one lane per centre, the wave's own row
      }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int64_t i = base + e * kQatThreads + threadIdx.x;
      if (i < n && grad_w) store_from_float(grad_w, gwdt, i, MODE == 0 ? (2.0f * g0) * gw[e] : gw[e]);
    }
  }
  if (KT > 0) {
    const float r = wave_sum16(sums);
    if ((lane & 3) == 0) red[wave][lane >> 2] = r;
  }
  __syncthreads();
  for (int j = threadIdx.x; j < K; j += kQatThreads) {
    const float s = (red[0][j] + red[1][j]) + (red[2][j] + red[3][j]);
    partial[static_cast<int64_t>(blockIdx.x) * K + j] = MODE == 0 ? -2.0f * g0 * s : s;
  }
}

// out[j] = scale * sum over the `rows` partial rows of column j: CW columns a
// work-group, 1024 / CW threads per column each adding every (1024 / CW)-th
// row, then a tree over them (a fixed order).  One thread per column adding
// row after row was a chain of `rows` dependent loads: at 2,304 rows 217 us on
// average over a training step's five calls, now 4 to 5 us.
template <int CW>
__global__ __launch_bounds__(1024) void qat_reduce_kernel(const float* __restrict__ partial, int64_t rows, int cols,
                                                          float scale, float* __restrict__ out) {
  __shared__ float red[1024];
  constexpr int R = 1024 / CW;
  const int col = blockIdx.x * CW + (threadIdx.x % CW), r0 = threadIdx.x / CW;
  float s = 0.0f;
  if (col < cols) {
#pragma unroll 4
    for (int64_t r = r0; r < rows; r += R) s += partial[r * cols + col];
  }
  red[threadIdx.x] = s;
#pragma unroll
  for (int h = R / 2; h >= 1; h >>= 1) {
    __syncthreads();
    if (r0 < h) red[threadIdx.x] += red[threadIdx.x + h * CW];
  }
  if (r0 == 0 && col < cols) out[col] = red[threadIdx.x] * scale;
}

void launch_reduce(const float* partial, int64_t rows, int cols, float scale, float* out, hipStream_t s) {
  if (cols == 1)
    hipLaunchKernelGGL(qat_reduce_kernel<1>, dim3(1), dim3(1024), 0, s, partial, rows, cols, scale, out);
  else
    hipLaunchKernelGGL(qat_reduce_kernel<16>, dim3((cols + 15) / 16), dim3(1024), 0, s, partial, rows, cols, scale,
                       out);
}

// (mean, sum of squared deviations from it) of each work-group's contiguous
// run of `per` weights: two passes over the run, the second from the caches.
// The separation kernel merges the runs, so the margin's std needs two
// launches where separate mean and variance reductions took five.
__global__ __launch_bounds__(kQatThreads) void moments_kernel(const void* __restrict__ w, int wdt, int64_t n,
                                                              int64_t per, float2* __restrict__ partial) {
  __shared__ float red[4];
  const int64_t lo = static_cast<int64_t>(blockIdx.x) * per, hi = lo + per < n ? lo + per : n;
  float mean = 0.0f;
#pragma unroll
  for (int pass = 0; pass < 2; ++pass) {
    float acc = 0.0f;
    for (int64_t base = lo; base < hi; base += kQatChunk) {
      int64_t at[kQatEpt];
      float v[kQatEpt];
#pragma unroll
      for (int e = 0; e < kQatEpt; ++e) {
        const int64_t i = base + e * kQatThreads + threadIdx.x;
        at[e] = i < hi ? i : hi - 1;
      }
      load_ept(w, wdt, at, v);
#pragma unroll
      for (int e = 0; e < kQatEpt; ++e)
        if (base + e * kQatThreads + threadIdx.x < hi) acc += pass ? (v[e] - mean) * (v[e] - mean) : v[e];
    }
    const float s = block_sum(acc, red);
    if (pass) {
      if (threadIdx.x == 0) partial[blockIdx.x] = make_float2(mean, s);
    } else {
      mean = s / static_cast<float>(hi - lo);
    }
  }
}

__device__ __forceinline__ double block_sum_f64(double v, double* red) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// Separation loss and its gradient in the centres (one work-group), after the
// runs' moments are merged (their count, mean and squared deviations, in
// double: a few values per thread):
//   delta = eta * 6 * max(sqrt(var), 1e-12) / K,
//   L = sum_{a<b} relu(delta - sqrt((c_a - c_b)^2 + eps))^2,
//   dL/dc_a = sum_{b != a} -2 relu(delta - r_ab) (c_a - c_b) / r_ab.
__global__ __launch_bounds__(kQatThreads) void separation_kernel(const float* __restrict__ c, int K,
                                                                 const float2* __restrict__ runs, int nruns,
                                                                 int64_t per, int64_t n, float eta, float eps,
                                                                 float* __restrict__ loss, float* __restrict__ grad_c) {
  __shared__ float cs[256];
  __shared__ float red[4];
  __shared__ double redd[4];
  for (int j = threadIdx.x; j < K; j += kQatThreads) cs[j] = c[j];
  double m = 0.0, v = 0.0;
  for (int r = threadIdx.x; r < nruns; r += kQatThreads) {
    const int64_t lo = r * per, len = (lo + per < n ? lo + per : n) - lo;
    m += static_cast<double>(len) * runs[r].x;
  }
  const double mean = block_sum_f64(m, redd) / static_cast<double>(n);
  for (int r = threadIdx.x; r < nruns; r += kQatThreads) {
    const int64_t lo = r * per, len = (lo + per < n ? lo + per : n) - lo;
    const double d = runs[r].x - mean;
    v += runs[r].y + static_cast<double>(len) * d * d;
  }
  const float var = static_cast<float>(block_sum_f64(v, redd) / static_cast<double>(n));
  const float sigma = fmaxf(sqrtf(var), 1e-12f);
  const float delta = eta * 6.0f * sigma / static_cast<float>(K);
  float acc = 0.0f;
  for (int a = threadIdx.x; a < K; a += kQatThreads) {
    float g = 0.0f;
    for (int b = 0; b < K; ++b) {
      if (b == a) continue;
      const float diff = cs[a] - cs[b];
      const float r = sqrtf(diff * diff + eps);
      const float h = fmaxf(delta - r, 0.0f);
      if (b > a) acc += h * h;
      g += -2.0f * h * diff / r;
    }
    if (grad_c) grad_c[a] = g;
  }
  const float s = block_sum(acc, red);
  if (threadIdx.x == 0) *loss = s;
}

inline int64_t qat_blocks(int64_t n) { return (n + kQatChunk - 1) / kQatChunk; }

inline int64_t qat_grid(int64_t n) {
  const int64_t b = qat_blocks(n), trips = (b + kQatMaxBlocks - 1) / kQatMaxBlocks;
  return b > 0 ? (b + trips - 1) / trips : 0;
}

// Work-groups of a backward: K <= 16 at most four per CU (within qat_blocks:
// half as many elements per trip as a chunk needs at least half as many).
inline int64_t qat_backward_grid(int64_t n, int K) {
  if (K > 16) return qat_grid(n);
  const int64_t b = qat_blocks(n), most = 4 * device_cus();
  return b < most ? b : most;
}

// The kernel instance of K centres.
template <class F>
void by_centres(int K, F f) {
  if (K == 4) f(std::integral_constant<int, 4>());
  else if (K == 8) f(std::integral_constant<int, 8>());
  else if (K == 16) f(std::integral_constant<int, 16>());
  else if (K < 16) f(std::integral_constant<int, kAnyTo16>());
  else f(std::integral_constant<int, 0>());
}

struct Taus {
  float tau, inv, il;
  explicit Taus(double t)
      : tau(static_cast<float>(t)), inv(static_cast<float>(1.0 / t)), il(static_cast<float>(kLog2e / t)) {}
};

}  // namespace
}  // namespace dimq

using namespace dimq;

extern "C" int64_t dimq_qat_workspace_bytes(int64_t n, int64_t n_centers) {
  if (n < 0 || n_centers < 1) return -1;
  const int64_t blocks = qat_blocks(n > 0 ? n : 1);
  return blocks * (n_centers > 1 ? n_centers : 1) * static_cast<int64_t>(sizeof(float)) + 256;
}

static int qat_check(const void* w, int w_dtype, int64_t n, const float* centers, int64_t K, double tau) {
  DIMQ_CHECK(w_dtype == DIMQ_F32 || w_dtype == DIMQ_F16 || w_dtype == DIMQ_BF16 || w_dtype == DIMQ_F64,
             "weights must be fp32, fp16, bf16 or fp64");
  DIMQ_CHECK(n >= 0, "the weight size must be non-negative");
  DIMQ_CHECK(n == 0 || w != nullptr, "weights are required");
  DIMQ_CHECK(centers != nullptr && K >= 1 && K <= 256, "centers must hold between 1 and 256 values");
  DIMQ_CHECK(tau > 0.0, "tau must be positive (the reference clamps it to at least 1e-12)");
  DIMQ_CHECK(qat_blocks(n) < (int64_t)1 << 31, "weights too large for one launch");
  return DIMQ_OK;
}

extern "C" int dimq_softmin_loss_forward(const void* w, int w_dtype, int64_t n, const float* centers, int64_t n_centers,
                                         double tau, int mean_reduction, float* aux, float* loss, void* workspace,
                                         int64_t workspace_bytes, void* stream) {
  int rc = qat_check(w, w_dtype, n, centers, n_centers, tau);
  if (rc != DIMQ_OK) return rc;
  DIMQ_CHECK(loss != nullptr, "loss output is required");
  DIMQ_CHECK(workspace != nullptr && workspace_bytes >= dimq_qat_workspace_bytes(n, n_centers),
             "workspace must hold dimq_qat_workspace_bytes bytes");
  const hipStream_t s = as_stream(stream);
  float* partial = static_cast<float*>(workspace);
  const int64_t blocks = qat_grid(n);
  if (n == 0) {
    launch_reduce(partial, 0, 1, 0.0f, loss, s);
    return check_launch("softmin loss");
  }
  const Taus t(tau);
  const int K = static_cast<int>(n_centers);
  by_centres(K, [&](auto kt) {
    hipLaunchKernelGGL((qat_forward_kernel<0, decltype(kt)::value>), dim3(static_cast<unsigned>(blocks)),
                       dim3(kQatThreads), 0, s, w, w_dtype, n, centers, K, t.inv, t.il, t.tau,
                       reinterpret_cast<float2*>(aux), partial, nullptr);
  });
  rc = check_launch("softmin loss");
  if (rc != DIMQ_OK) return rc;
  launch_reduce(partial, blocks, 1, mean_reduction ? 1.0f / static_cast<float>(n) : 1.0f, loss, s);
  return check_launch("softmin loss (sum)");
}

extern "C" int dimq_softmin_loss_backward(const void* w, int w_dtype, int64_t n, const float* centers,
                                          int64_t n_centers, double tau, int mean_reduction, const float* aux,
                                          const float* grad_loss, void* grad_w, int grad_w_dtype, float* grad_centers,
                                          void* workspace, int64_t workspace_bytes, void* stream) {
  int rc = qat_check(w, w_dtype, n, centers, n_centers, tau);
  if (rc != DIMQ_OK) return rc;
  DIMQ_CHECK(aux != nullptr && grad_loss != nullptr, "the forward's aux and the loss gradient are required");
  DIMQ_CHECK(grad_w == nullptr || is_float_dtype(grad_w_dtype), "grad_w must be floating point");
  DIMQ_CHECK(grad_centers != nullptr, "grad_centers is required");
  DIMQ_CHECK(workspace != nullptr && workspace_bytes >= dimq_qat_workspace_bytes(n, n_centers),
             "workspace must hold dimq_qat_workspace_bytes bytes");
  DIMQ_CHECK(!mean_reduction, "the mean reduction's backward is the sum's scaled by 1/n: pass the scaled gradient");
  const hipStream_t s = as_stream(stream);
  float* partial = static_cast<float*>(workspace);
  const int K = static_cast<int>(n_centers);
  const int64_t blocks = qat_backward_grid(n, K);
  const Taus t(tau);
  if (blocks > 0) {
    by_centres(K, [&](auto kt) {
      hipLaunchKernelGGL((qat_backward_kernel<0, decltype(kt)::value>), dim3(static_cast<unsigned>(blocks)),
                         dim3(kQatThreads), 0, s, w, w_dtype, n, centers, K, t.inv, t.il,
                         reinterpret_cast<const float2*>(aux), grad_loss, nullptr, 0, grad_w, grad_w_dtype, partial);
    });
    rc = check_launch("softmin loss backward");
    if (rc != DIMQ_OK) return rc;
  }
  launch_reduce(partial, blocks, K, 1.0f, grad_centers, s);
  return check_launch("softmin loss backward (centres)");
}

extern "C" int dimq_soft_dequantize_forward(const void* w, int w_dtype, int64_t n, const float* centers,
                                            int64_t n_centers, double tau, void* out, float* aux, void* stream) {
  int rc = qat_check(w, w_dtype, n, centers, n_centers, tau);
  if (rc != DIMQ_OK) return rc;
  DIMQ_CHECK(n == 0 || (out != nullptr && aux != nullptr), "out and aux are required");
  if (n == 0) return DIMQ_OK;
  const Taus t(tau);
  const int K = static_cast<int>(n_centers);
  by_centres(K, [&](auto kt) {
    hipLaunchKernelGGL((qat_forward_kernel<1, decltype(kt)::value>), dim3(static_cast<unsigned>(qat_grid(n))),
                       dim3(kQatThreads), 0, as_stream(stream), w, w_dtype, n, centers, K, t.inv, t.il, t.tau,
                       reinterpret_cast<float2*>(aux), nullptr, out);
  });
  return check_launch("soft dequantize");
}

extern "C" int dimq_soft_dequantize_backward(const void* w, int w_dtype, int64_t n, const float* centers,
                                             int64_t n_centers, double tau, const float* aux, const void* grad_out,
                                             int grad_out_dtype, void* grad_w, int grad_w_dtype, float* grad_centers,
                                             void* workspace, int64_t workspace_bytes, void* stream) {
  int rc = qat_check(w, w_dtype, n, centers, n_centers, tau);
  if (rc != DIMQ_OK) return rc;
  DIMQ_CHECK(n == 0 || (aux != nullptr && grad_out != nullptr), "the forward's aux and grad_out are required");
  DIMQ_CHECK(is_float_dtype(grad_out_dtype), "grad_out must be floating point");
  DIMQ_CHECK(grad_w == nullptr || is_float_dtype(grad_w_dtype), "grad_w must be floating point");
  DIMQ_CHECK(grad_centers != nullptr, "grad_centers is required");
  DIMQ_CHECK(workspace != nullptr && workspace_bytes >= dimq_qat_workspace_bytes(n, n_centers),
             "workspace must hold dimq_qat_workspace_bytes bytes");
  const hipStream_t s = as_stream(stream);
  float* partial = static_cast<float*>(workspace);
  const int K = static_cast<int>(n_centers);
  const int64_t blocks = qat_backward_grid(n, K);
  const Taus t(tau);
  if (blocks > 0) {
    by_centres(K, [&](auto kt) {
      hipLaunchKernelGGL((qat_backward_kernel<1, decltype(kt)::value>), dim3(static_cast<unsigned>(blocks)),
                         dim3(kQatThreads), 0, s, w, w_dtype, n, centers, K, t.inv, t.il,
                         reinterpret_cast<const float2*>(aux), nullptr, grad_out, grad_out_dtype, grad_w, grad_w_dtype, partial);
    });
    rc = check_launch("soft dequantize backward");
    if (rc != DIMQ_OK) return rc;
  }
  launch_reduce(partial, blocks, K, 1.0f, grad_centers, s);
  return check_launch("soft dequantize backward (centres)");
}

extern "C" int dimq_separation_loss(const void* w, int w_dtype, int64_t n, const float* centers, int64_t n_centers,
                                    double eta, double eps, float* loss, float* grad_centers, void* workspace,
                                    int64_t workspace_bytes, void* stream) {
  int rc = qat_check(w, w_dtype, n, centers, n_centers, 1.0);
  if (rc != DIMQ_OK) return rc;
  DIMQ_CHECK(n >= 1, "separation_loss needs a non-empty weight (its margin is a multiple of std(w))");
  DIMQ_CHECK(loss != nullptr, "loss output is required");
  DIMQ_CHECK(workspace != nullptr && workspace_bytes >= dimq_qat_workspace_bytes(n, n_centers),
             "workspace must hold dimq_qat_workspace_bytes bytes");
  DIMQ_CHECK(eps >= 0.0, "eps must be non-negative");
  const hipStream_t s = as_stream(stream);
  // runs of at least 2,048 weights (8 bytes each: within 4 bytes per 1,024 plus the 256 spare)
  int64_t per = 2 * kQatChunk;
  if ((n + per - 1) / per > kQatMaxBlocks) per = (n + kQatMaxBlocks - 1) / kQatMaxBlocks;
  const int64_t runs = (n + per - 1) / per;
  float2* partial = static_cast<float2*>(workspace);
  hipLaunchKernelGGL(moments_kernel, dim3(static_cast<unsigned>(runs)), dim3(kQatThreads), 0, s, w, w_dtype, n, per,
                     partial);
  rc = check_launch("separation loss (moments)");
  if (rc != DIMQ_OK) return rc;
  hipLaunchKernelGGL(separation_kernel, dim3(1), dim3(kQatThreads), 0, s, centers, static_cast<int>(n_centers),
                     partial, static_cast<int>(runs), per, n, static_cast<float>(eta), static_cast<float>(eps), loss,
                     grad_centers);
  return check_launch("separation loss");
}
