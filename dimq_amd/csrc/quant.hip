// Element-wise quantization kernels:
//  * u4 activation quantization (dimq_backend/reference.py:11-21,
//    csrc/dimq_pack.cu:37-48) with an IEEE divide and round-half-to-even;
//  * activation x centroid product tables (dimq_backend/reference.py:32-44,
//    csrc/dimq_product_table.cu:11-25), per layer or per output channel;
//  * nearest-centre index assignment (quant/dimq.py:197-221,
//    dimq_backend/export.py:24-35), per layer or per output channel.
#include "common.h"

namespace dimq {
namespace {

constexpr int kThreads = 256;

// 8 activations per thread; the HIP divide is IEEE-correct (no fast-math).
__global__ __launch_bounds__(kThreads) void quantize_act_kernel(const void* __restrict__ x, int dt, int64_t n,
                                                                float s, int zp, uint8_t* __restrict__ out) {
  const int64_t base = (static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x) * 8;
  if (base >= n) return;
  if (base + 8 <= n) {
    uint32_t lo = 0, hi = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t q = (uint32_t)quantize_u4(load_as_float(x, dt, base + j), s, zp);
      if (j < 4) lo |= q << (8 * j); else hi |= q << (8 * (j - 4));
    }
    if (((reinterpret_cast<uintptr_t>(out) + base) & 7) == 0) {
      *reinterpret_cast<uint2*>(out + base) = make_uint2(lo, hi);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) out[base + j] = (uint8_t)((j < 4 ? lo >> (8 * j) : hi >> (8 * (j - 4))) & 0xff);
    }
  } else {
    for (int64_t i = base; i < n; ++i) out[i] = (uint8_t)quantize_u4(load_as_float(x, dt, i), s, zp);
  }
}

// W4A4 activations for the weight-only kernels: out = fp16(q - zp) with
// q = clamp(rint(x / s) + zp, 0, 15), the same code as quantize_act_kernel.
// q - zp is an integer in [-15, 15], exact in fp16, so a weight-only GEMM/conv
// over these values times s equals sum_k C[w] * (s * (a - zp)) up to fp32
// summation order.  kQa4Groups groups of 8 activations per thread, group u of
// thread t of work-group b at (b * kQa4Groups + u) * kThreads + t (loads
// coalesced per u, all of a thread's loads in flight at once); VEC: x is
// 16-byte aligned (vector loads of the 8 inputs).
template <int XT, bool VEC>
__global__ __launch_bounds__(kThreads) void quantize_a4_f16_kernel(const void* __restrict__ x, int64_t n, float s,
                                                                   int zp, uint16_t* __restrict__ out) {
  quantize_a4_f16_groups<XT, VEC, kQa4Groups>(
      x, n, s, zp, out, static_cast<int64_t>(blockIdx.x) * kThreads * kQa4Groups + threadIdx.x, kThreads);
}

// table[g][w][a] = C[g][w] * (s * (a - zp)), fp32, same operation order as
// the reference (product of the centroid and the dequantized level).
__global__ __launch_bounds__(kThreads) void product_table_kernel(const void* __restrict__ cb, int dt, int64_t total,
                                                                 float s, int zp, float* __restrict__ table) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x;
  if (i >= total) return;
  const int a = static_cast<int>(i & 15);
  const float w = load_as_float(cb, dt, i >> 4);
  const float ahat = s * static_cast<float>(a - zp);
  table[i] = w * ahat;
}

// Nearest centre with torch's argmin semantics on fp32 distances
// d(c) = RN(RN(x - c)^2) (quant/dimq.py:213-214): the first minimum wins, a
// NaN distance beats every number and the first NaN is kept.
//
// RN is monotone, so for a finite x, d(c) does not increase as c rises
// towards x and does not decrease as c rises beyond it: over the centres in
// ascending order the minimum sits at one of x's two neighbours, and the
// centres with that distance form one run around them.  The work-group sorts
// its row's centres in LDS once (rank sort on (value, index)), and each
// element costs a binary search, two distances and a scan of the tied run
// (usually one step), whatever the number of centres.  NaN distances come
// only from NaN centres, a NaN x, or an infinite x meeting the same
// infinity; those cases are answered from the first-index flags below.
struct CentreRow {
  float sv[256];  // centres in ascending order (ties by index)
  int si[256];    // their indices
  __attribute__((aligned(16))) float raw[256];  // WIDE: padded to a multiple of 4 with +inf
  int first_nan, first_pinf, first_ninf;  // first NaN / +inf / -inf centre, K if none
};

__device__ __forceinline__ float centre_dist(float x, float c) {
#pragma clang fp contract(off)  // one rounding of the square, never fused into a later add
  const float diff = x - c;
  return diff * diff;
}

// Whole work-group: the row's K (1..256) centres into `r`.
// WIDE: the ranks from four centres per LDS read (4,096 x 4,096 weights, 64 and
// 256 centres per row: 43.5 -> 42.1 and 84.6 -> 78.9 us; but 20,000 rows of 9,
// where the set-up is most of the time, 29 -> 38 at 17 centres).
template <bool WIDE>
__device__ void centre_row_setup(const float* __restrict__ c, int K, CentreRow& r) {
  if (threadIdx.x == 0) {
    r.first_nan = K;
    r.first_pinf = K;
    r.first_ninf = K;
  }
  const int K4 = WIDE ? (K + 3) & ~3 : K;
  for (int j = threadIdx.x; j < K4; j += blockDim.x) r.raw[j] = j < K ? c[j] : __builtin_inff();
  __syncthreads();
  for (int j = threadIdx.x; j < K; j += blockDim.x) {
    const float v = r.raw[j];
    if (v != v) atomicMin(&r.first_nan, j);
    if (v == __builtin_inff()) atomicMin(&r.first_pinf, j);
    if (v == -__builtin_inff()) atomicMin(&r.first_ninf, j);
    int rank = 0;
#pragma unroll 8
    for (int i = 0; i < K4; i += WIDE ? 4 : 1) {  // a padded entry is never below v, nor equal to it ahead of j
      if constexpr (WIDE) {
        const float4 u = *reinterpret_cast<const float4*>(&r.raw[i]);
        rank += ((u.x < v) || (u.x == v && i < j)) + ((u.y < v) || (u.y == v && i + 1 < j)) +
                ((u.z < v) || (u.z == v && i + 2 < j)) + ((u.w < v) || (u.w == v && i + 3 < j));
      } else {
        const float u = r.raw[i];
        rank += (u < v) || (u == v && i < j);
      }
    }
    // with a NaN centre ranks can collide; the sorted view is then unused
    r.sv[rank] = v;
    r.si[rank] = j;
  }
  __syncthreads();
}

__device__ __forceinline__ int nearest_centre(float x, const CentreRow& r, int K) {
  if (x != x) return 0;  // every distance NaN
  if (x == __builtin_inff() || x == -__builtin_inff()) {
    // NaN distances: the NaN centres and the centres equal to x; else all inf
    const int f = min(r.first_nan, x > 0.0f ? r.first_pinf : r.first_ninf);
    return f < K ? f : 0;
  }
  if (r.first_nan < K) return r.first_nan;
  int pos = 0;  // number of centres <= x
#pragma unroll
  for (int step = 256; step > 0; step >>= 1)
    if (pos + step <= K && r.sv[pos + step - 1] <= x) pos += step;
  const int L = pos - 1, R = pos;
  const float dl = L >= 0 ? centre_dist(x, r.sv[L]) : 0.0f;
  const float dr = R < K ? centre_dist(x, r.sv[R]) : 0.0f;
  const float ds = L < 0 ? dr : (R >= K ? dl : fminf(dl, dr));
  int best = K;
  if (L >= 0 && dl == ds)
    for (int i = L; i >= 0 && centre_dist(x, r.sv[i]) == ds; --i) best = min(best, r.si[i]);
  if (R < K && dr == ds)
    for (int i = R; i < K && centre_dist(x, r.sv[i]) == ds; ++i) best = min(best, r.si[i]);
  return best;
}

// E elements of a row: four consecutive ones (VEC: the row is aligned for one
// load of all four) or E that lie kThreads apart; past the row's end the last
// one again.
template <bool VEC, int E>
__device__ __forceinline__ void load_some(const void* __restrict__ w, int dt, int64_t base, int64_t k, int64_t row_len,
                                          float (&x)[E]) {
  if constexpr (VEC) {
    const int64_t e = base + (k < row_len ? k : row_len - 4);
    if (dt == DIMQ_F32) {
      const float4 t = *reinterpret_cast<const float4*>(static_cast<const float*>(w) + e);
      x[0] = t.x; x[1] = t.y; x[2] = t.z; x[3] = t.w;
    } else {
      const uint2 t = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(w) + e);
      const uint32_t h[4] = {t.x & 0xffffu, t.x >> 16, t.y & 0xffffu, t.y >> 16};
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = dt == DIMQ_F16 ? f16_bits_to_float(h[i]) : bf16_bits_to_float(h[i]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const int64_t kk = k + i * kThreads;
      x[i] = load_as_float(w, dt, base + (kk < row_len ? kk : row_len - 1));
    }
  }
}

template <bool VEC, int E>
__device__ __forceinline__ void store_some(uint8_t* __restrict__ idx, void* __restrict__ values, int dt, int64_t base,
                                           int64_t k, int64_t row_len, const int (&j)[E], const float (&v)[E]) {
  if constexpr (VEC) {
    if (k >= row_len) return;
    if (idx) *reinterpret_cast<uint32_t*>(idx + base + k) = j[0] | (j[1] << 8) | (j[2] << 16) | (j[3] << 24);
    if (!values) return;
    if (dt == DIMQ_F32) {
      *reinterpret_cast<float4*>(static_cast<float*>(values) + base + k) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
      uint32_t h[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) h[i] = dt == DIMQ_F16 ? float_to_f16_bits(v[i]) : float_to_bf16_bits(v[i]);
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(values) + base + k) =
          make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
    }
  } else {
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const int64_t kk = k + i * kThreads;
      if (kk >= row_len) return;
      if (idx) idx[base + kk] = static_cast<uint8_t>(j[i]);
      if (values) store_from_float(values, dt, base + kk, v[i]);
    }
  }
}

// Nearest-centre assignment of a [rows, row_len] tensor (per_channel: row r
// uses centres[r * K ..]; else one set for all).  One work-group per segment
// of a row, E elements per thread and trip (their chains interleave; VEC: one
// load, one index store and one value store for all four); writes the
// index (idx, nullable) and / or centres[idx].to(dtype) (values, nullable).
// hard_quantize_weight, quant/dimq.py:197-221.
//
// KD = 4, 8 (K <= KD): the first minimum of the K distances directly, centres
// in scalar registers (5 VALU per centre; padded with the last centre, which
// is never nearer than itself).  With finite centres a NaN or infinite element
// finds no distance below the first and takes index 0, as torch's argmin.
// KD = 16, 256: the sorted centres, log2 KD search steps in LDS, then the two
// neighbours' distances.  They decide unless a further centre's rounded
// distance can equal theirs: with every centre finite and neighbours at least
// g apart, a centre c1 beyond c2 at distance a from x has (a + g) / a >= 1 +
// 2^-19 for a < 2^19 g, two roundings of 2^-24 cannot close that, and with
// 1e-18 < g and a < 1e18 no square under- or overflows.  Elements outside that
// bound, NaN and infinite ones take the full scan.
// KD = 0 (one element per thread): the sorted centres and, for every element,
// the search and scan; the bound costs more to set up than it saves there.
// 4,096 x 4,096 fp32 weights, 8 centres per row: 97.8 -> 29.5 us; 16:
// 98.9 -> 33.1; 256: 129.1 -> 89.2; a plain copy of as many bytes 30.
template <int KD, bool VEC, int E>
__global__ __launch_bounds__(kThreads) void nearest_centre_kernel(const void* __restrict__ w, int dt, int64_t row_len,
                                                                  const float* __restrict__ centers, int K,
                                                                  int per_channel, uint8_t* __restrict__ idx,
                                                                  void* __restrict__ values, int64_t seg_per_row,
                                                                  int trips) {
  __shared__ CentreRow r;
  __shared__ int gap;
  const int64_t row = static_cast<uint32_t>(blockIdx.x) / static_cast<uint32_t>(seg_per_row);
  const int64_t seg = static_cast<int64_t>(blockIdx.x) - row * seg_per_row;
  static_assert(!VEC || E == 4, "one load of four elements");
  constexpr int kTrip = E * kThreads;
  const int64_t base = row * row_len;
  const float* cr = centers + (per_channel ? row * K : 0);
  int64_t k = seg * kTrip * trips + (VEC ? 4 * threadIdx.x : threadIdx.x);
  float xn[E];
  load_some<VEC, E>(w, dt, base, k, row_len, xn);  // before the centres are looked at
  bool fast = true;     // KD <= 8: every centre finite
  float limit = 0.0f;   // KD > 8: the bound above, 0 when the scan is always needed
  float c[KD > 0 && KD <= 8 ? KD : 1];
  if constexpr (KD == 0) {
    centre_row_setup<false>(cr, K, r);
    for (int t = 0; t < trips && k < row_len; ++t, k += kTrip) {
      if (t > 0) load_some<VEC, E>(w, dt, base, k, row_len, xn);
      const int j[1] = {nearest_centre(xn[0], r, K)};
      const float v[1] = {r.raw[j[0]]};
      store_some<VEC, E>(idx, values, dt, base, k, row_len, j, v);
    }
    return;
  }
  if constexpr (KD <= 8) {
#pragma unroll
    for (int j = 0; j < KD; ++j) {
      c[j] = cr[j < K ? j : K - 1];
      fast &= __builtin_isfinite(c[j]);
    }
    if (!fast) centre_row_setup<true>(cr, K, r);
  } else {
    if (threadIdx.x == 0) gap = __float_as_int(__builtin_inff());
    centre_row_setup<true>(cr, K, r);
    bool fin = true;
    float mine = __builtin_inff();
    static_assert(KD <= kThreads, "one sorted centre per thread");
    if (const int j = threadIdx.x; j < KD) {
      if (j >= K) r.sv[j] = __builtin_inff();
      else fin = __builtin_isfinite(r.sv[j]);
      if (j + 1 < K) {
        const float g = r.sv[j + 1] - r.sv[j];
        mine = g > 0.0f ? g : 0.0f;
      }
    }
    if (threadIdx.x < 64 || KD > 64) {  // whole waves
#pragma unroll
      for (int m = 32; m >= 1; m >>= 1) mine = fminf(mine, __shfl_xor(mine, m, 64));
      if ((threadIdx.x & 63) == 0) atomicMin(&gap, __float_as_int(mine));  // positive floats order as their bits
    }
    fin = __syncthreads_and(fin);  // r.first_nan covers rows whose sorted view a NaN spoils
    const float g = __int_as_float(gap);
    limit = fin && r.first_nan >= K && g > 1e-18f ? fminf(g * 524288.0f, 1e18f) : 0.0f;
  }
  for (int t = 0; t < trips; ++t, k += kTrip) {
    float x[E], v[E];
    int best[E];
#pragma unroll
    for (int i = 0; i < E; ++i) x[i] = xn[i];
    if (t + 1 < trips) load_some<VEC, E>(w, dt, base, k + kTrip, row_len, xn);
    if constexpr (KD <= 8) {
      if (fast) {
        float d[E];
#pragma unroll
        for (int i = 0; i < E; ++i) {
          d[i] = centre_dist(x[i], c[0]);
          best[i] = 0;
          v[i] = c[0];
        }
#pragma unroll
        for (int j = 1; j < KD; ++j)
#pragma unroll
          for (int i = 0; i < E; ++i) {
            const float dj = centre_dist(x[i], c[j]);
            const bool less = dj < d[i];
            d[i] = less ? dj : d[i];
            best[i] = less ? j : best[i];
            v[i] = less ? c[j] : v[i];
          }
      } else {
#pragma unroll
        for (int i = 0; i < E; ++i) {
          best[i] = nearest_centre(x[i], r, K);
          v[i] = r.raw[best[i]];
        }
      }
    } else {
      int pos[E];  // the last centre <= x, or 0
#pragma unroll
      for (int i = 0; i < E; ++i) pos[i] = 0;
#pragma unroll
      for (int step = KD / 2; step > 0; step >>= 1)
#pragma unroll
        for (int i = 0; i < E; ++i) pos[i] += r.sv[pos[i] + step] <= x[i] ? step : 0;  // sv is +inf from K on
      bool scan[E];
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const int nx = pos[i] + 1 < KD ? pos[i] + 1 : pos[i];
        const float lo = r.sv[pos[i]], hi = r.sv[nx];
        const int jl = r.si[pos[i]], jh = nx < K ? r.si[nx] : 256;
        const float dl = centre_dist(x[i], lo), dh = centre_dist(x[i], hi);
        const bool up = dh < dl || (dh == dl && jh < jl);
        best[i] = up ? jh : jl;
        v[i] = up ? hi : lo;
        scan[i] = !(fabsf(x[i] - v[i]) < limit);
      }
#pragma unroll
      for (int i = 0; i < E; ++i)
        if (scan[i]) {
          best[i] = nearest_centre(x[i], r, K);
          v[i] = r.raw[best[i]];
        }
    }
    store_some<VEC, E>(idx, values, dt, base, k, row_len, best, v);
  }
}

template <bool VEC, int E>
void launch_nearest_form(const void* w, int dt, int64_t row_len, const float* centers, int K, int per_channel,
                         uint8_t* idx, void* values, int64_t seg, int trips, unsigned blocks, hipStream_t st) {
#define DIMQ_NEAREST(KD)                                                                                            \
  hipLaunchKernelGGL((nearest_centre_kernel<KD, VEC, E>), dim3(blocks), dim3(kThreads), 0, st, w, dt, row_len,      \
                     centers, K, per_channel, idx, values, seg, trips)
  if (K <= 4) DIMQ_NEAREST(4);
  else if (K <= 8) DIMQ_NEAREST(8);
  else if constexpr (E == 1) DIMQ_NEAREST(0);
  else if (K <= 16) DIMQ_NEAREST(16);
  else DIMQ_NEAREST(256);
#undef DIMQ_NEAREST
}

int launch_nearest_centre(const void* w, int dt, int64_t rows, int64_t row_len, const float* centers, int K,
                          int per_channel, uint8_t* idx, void* values, hipStream_t st) {
  if (rows == 0 || row_len == 0) return DIMQ_OK;
  const int pc = per_channel ? 1 : 0;
  const int64_t quads = (row_len + 4 * kThreads - 1) / (4 * kThreads);  // work-groups of a row at four elements a thread
  // One element per thread and trip: a small tensor (four times the
  // work-groups), and short rows, where each work-group's time is the set-up
  // (20,000 rows of 9: 9 centres 41 us on the four-element form, 19 here, 64
  // centres 82 and 34; rows of 256 41 and 31, 64 and 47; of 300, 17 centres 51
  // and 47; of 512 52 and 59; up to 8 centres, whose set-up is a load, rows of
  // 9 30 and 22, of 256 28 and 31).
  const int64_t one = K > 16 ? 352 : K > 8 ? kThreads : 64;
  if (rows * quads < device_cus() || row_len <= one) {
    const int trips = row_len <= one && row_len > kThreads && rows * quads >= device_cus() ? 2 : 1;
    const int64_t seg = (row_len + kThreads * trips - 1) / (kThreads * trips);
    DIMQ_CHECK(rows * seg < (int64_t)1 << 31, "tensor too large for one launch");
    launch_nearest_form<false, 1>(w, dt, row_len, centers, K, pc, idx, values, seg, trips,
                                  static_cast<unsigned>(rows * seg), st);
    return check_launch("nearest centre");
  }
  // trips per work-group: 1 while that leaves fewer than 4096 work-groups, up
  // to 4 for large tensors (the centres are set up once per work-group)
  int trips = 1;
  while (trips < 4 && rows * ((quads + trips - 1) / trips) >= 4096 && quads > trips) trips *= 2;
  const int64_t seg = (quads + trips - 1) / trips;
  DIMQ_CHECK(rows * seg < (int64_t)1 << 31, "tensor too large for one launch");
  const bool vec = row_len % 4 == 0 && aligned(w, 4 * dtype_size(dt)) && (idx == nullptr || aligned(idx, 4)) &&
                   (values == nullptr || aligned(values, 4 * dtype_size(dt)));
  const unsigned blocks = static_cast<unsigned>(rows * seg);
  if (vec) launch_nearest_form<true, 4>(w, dt, row_len, centers, K, pc, idx, values, seg, trips, blocks, st);
  else launch_nearest_form<false, 4>(w, dt, row_len, centers, K, pc, idx, values, seg, trips, blocks, st);
  return check_launch("nearest centre");
}

}  // namespace

// Activation codebook (the QAT wrapper's activation_centers,
// quant/dimq_wrapper.py:80-85 via hard_quantize_weight, quant/dimq.py:197-221):
// out = C_a[argmin_c (x - C_a[c])^2] in x's dtype (K in [1, 256]).
int launch_act_codebook(const void* x, int x_dtype, int64_t n, const float* centers, int K, void* out,
                        hipStream_t st) {
  return launch_nearest_centre(x, x_dtype, 1, n, centers, K, 0, nullptr, out, st);
}

// Launches quantize_a4_f16_kernel; out must be 16-byte aligned.
int launch_quantize_a4_f16(const void* x, int x_dtype, int64_t n, float s, int zp, uint16_t* out, hipStream_t st) {
  if (n == 0) return DIMQ_OK;
  const int64_t blocks = ((n + 7) / 8 + kThreads * kQa4Groups - 1) / (kThreads * kQa4Groups);
  const bool vec = aligned(x, 16);
  const dim3 grid(static_cast<unsigned>(blocks));
#define DIMQ_QA4(XT)                                                                                 \
  if (vec)                                                                                           \
    hipLaunchKernelGGL((quantize_a4_f16_kernel<XT, true>), grid, dim3(kThreads), 0, st, x, n, s, zp, out); \
  else                                                                                               \
    hipLaunchKernelGGL((quantize_a4_f16_kernel<XT, false>), grid, dim3(kThreads), 0, st, x, n, s, zp, out)
  switch (x_dtype) {
    case DIMQ_F32: DIMQ_QA4(DIMQ_F32); break;
    case DIMQ_F16: DIMQ_QA4(DIMQ_F16); break;
    case DIMQ_BF16: DIMQ_QA4(DIMQ_BF16); break;
    default: hipLaunchKernelGGL((quantize_a4_f16_kernel<DIMQ_F64, false>), grid, dim3(kThreads), 0, st, x, n, s, zp,
                                out); break;
  }
#undef DIMQ_QA4
  return check_launch("quantize activations (W4A4 fast path)");
}

}  // namespace dimq

using namespace dimq;

// The W4A4 input form of a tensor: out = fp16(q - zp), q the reference's u4
// code (reference.py:11-21).  Entry point of a chain of W4A4 layers whose
// later inputs come from the quantizing epilogue of the layer before.
extern "C" int dimq_quantize_activation_f16(const void* x, int x_dtype, int64_t numel, double act_scale,
                                            int64_t act_zp, uint16_t* out, void* stream) {
  DIMQ_CHECK(is_float_dtype(x_dtype), "quantize_activation expects floating input");
  DIMQ_CHECK(act_scale > 0.0, "act_scale must be positive");
  DIMQ_CHECK(act_zp >= 0 && act_zp <= 15, "act_zero_point must be in [0, 15]");
  DIMQ_CHECK(numel >= 0, "numel must be non-negative");
  DIMQ_CHECK(aligned(out, 16), "out must be 16-byte aligned");
  return launch_quantize_a4_f16(x, x_dtype, numel, static_cast<float>(act_scale), static_cast<int>(act_zp), out,
                                as_stream(stream));
}

extern "C" int dimq_quantize_activation_u4(const void* x, int x_dtype, int64_t numel, double act_scale,
                                           int64_t act_zp, uint8_t* out, void* stream) {
  DIMQ_CHECK(is_float_dtype(x_dtype), "quantize_activation_u4 expects floating input");
  DIMQ_CHECK(act_scale > 0.0, "act_scale must be positive");
  DIMQ_CHECK(act_zp >= 0 && act_zp <= 15, "act_zero_point must be in [0, 15]");
  DIMQ_CHECK(numel >= 0, "numel must be non-negative");
  if (numel == 0) return DIMQ_OK;
  const int64_t threads_needed = (numel + 7) / 8;
  const int64_t blocks = (threads_needed + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(quantize_act_kernel, dim3((unsigned)blocks), dim3(kThreads), 0, as_stream(stream), x, x_dtype,
                     numel, static_cast<float>(act_scale), static_cast<int>(act_zp), out);
  return check_launch("quantize_activation_u4");
}

extern "C" int dimq_build_product_table_grouped(const void* codebook, int cb_dtype, int64_t groups, int64_t kc,
                                                double act_scale, int64_t act_zp, float* table, void* stream) {
  DIMQ_CHECK(is_float_dtype(cb_dtype), "build_product_table expects floating codebook");
  DIMQ_CHECK(act_scale > 0.0, "act_scale must be positive");
  DIMQ_CHECK(act_zp >= 0 && act_zp <= 15, "act_zero_point must be in [0, 15]");
  DIMQ_CHECK(groups >= 0 && kc > 0, "codebook shape must be positive");
  const int64_t total = groups * kc * 16;
  if (total == 0) return DIMQ_OK;
  const int64_t blocks = (total + kThreads - 1) / kThreads;
  hipLaunchKernelGGL(product_table_kernel, dim3((unsigned)blocks), dim3(kThreads), 0, as_stream(stream), codebook,
                     cb_dtype, total, static_cast<float>(act_scale), static_cast<int>(act_zp), table);
  return check_launch("build_product_table");
}

extern "C" int dimq_build_product_table(const void* codebook, int cb_dtype, int64_t cb_numel, double act_scale,
                                        int64_t act_zp, float* table, void* stream) {
  DIMQ_CHECK(is_float_dtype(cb_dtype), "build_product_table expects floating codebook");
  DIMQ_CHECK(cb_numel == 16, "build_product_table expects exactly 16 codebook entries");
  return dimq_build_product_table_grouped(codebook, cb_dtype, 1, 16, act_scale, act_zp, table, stream);
}

extern "C" int dimq_hard_quantize(const void* w, int w_dtype, int64_t rows, int64_t row_len, const float* centers,
                                  int64_t n_centers, int per_channel, uint8_t* indices, void* values, void* stream) {
  DIMQ_CHECK(w_dtype == DIMQ_F32 || w_dtype == DIMQ_F16 || w_dtype == DIMQ_BF16,
             "hard_quantize expects fp32/fp16/bf16 weights");
  DIMQ_CHECK(n_centers > 0, "centers must be non-empty");
  DIMQ_CHECK(n_centers <= 256, "at most 256 centers are supported (uint8 indices), got %lld",
             (long long)n_centers);
  DIMQ_CHECK(rows >= 0 && row_len >= 0, "weight shape must be non-negative");
  return launch_nearest_centre(w, w_dtype, rows, row_len, centers, static_cast<int>(n_centers), per_channel,
                               indices, values, as_stream(stream));
}
