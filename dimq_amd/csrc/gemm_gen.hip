// General pre-laid GEMM: the codebook Linear and Conv2d calls that no
// shape-specific kernel takes (channel counts off the tiles, NCHW or fp32 /
// bf16 convolutions, groups, dilation, 8-bit codebooks, K off the k steps,
// W4A4 layers), as
//
//   1. gen_prep_kernel: the packed indices and codebook rows -> W_hat as fp16
//      [rows][kp], k = (tap, channel) with the channels of a tap padded to a
//      multiple of 8 and the whole row to a k stage, each row scaled by the
//      power of two of the register-codebook kernels (decode.h) with the
//      factor in rs; and the activations -> fp16 rows of a pixel's channels
//      (transposed from NCHW through LDS, converted, or quantized to the
//      W4A4 codes a - zp), with the range guard's flags for fp32 / bf16.
//      fp16 channels-last (or row-major) activations whose channel count is
//      a multiple of 8 are read in place.
//   2. gen_gemm_kernel: an fp16 GEMM whose operands reach LDS through
//      global_load_lds in a ring of 64-k stages, after gemm_pd.hip's.  A lane's
//      16-byte chunk is 8 channels of one tap of one output pixel: its
//      address is formed per stage from the lane's running (tap, channel),
//      and chunks outside the image or past the last tap come from a zeroed
//      16 bytes in the workspace.
//   3. split_reduce_kernel, when the k range is split: adds the fp32 partial
//      outputs in a fixed order, then bias and epilogue.
//
// Before this path the calls ran on gemm_cb_kernel, which decodes every weight
// again in every 64-row tile and gathers each activation by itself: W4A4
// conv2d_lut, 32 x 256 x 14 x 14, 256 3x3 filters, 232 us.
#include "gemm_big.h"
#include "gemm_gen.h"

namespace dimq {
namespace {

constexpr int kGenCH = 8;             // 16-byte chunks of a stage row
constexpr int kGenK = 8 * kGenCH;     // k of a stage; a weight row is padded to whole stages
constexpr int kGenB = 64;             // rows and columns of a GEMM tile
constexpr int kGenS = 3;              // slots of the LDS ring
constexpr int kGenRows = 4;           // weight rows per work-group of the first launch, one per wave
constexpr int kGenRaw = 16384;        // packed bytes of a work-group's rows kept in LDS
constexpr int kGenPix = 64, kGenChan = 64;  // pixels x channels of an NCHW transpose work-group
// Laid-out activations and flags of a call in its workspace: larger ones go in
// several passes of whole images (Linear: rows) over the same workspace.  A
// depthwise layer's channels are padded eightfold, so its layout is 8 to 10
// times an fp16 input: 128 x 96 x 112 x 112, 3x3, needed 2.87 GiB in one pass.
// That layer takes 28.1 ms in ten passes (fp16, channels last; 29.3 in one, 257
// on gemm_cb_kernel) and 22.2 in 12 (fp32 NCHW; 22.3, 273).
constexpr int64_t kGenActBytes = 256ll << 20;

// Chunk c of stage row r lies at 128 r + ((c ^ gen_swz(r)) << 4), so that the
// 16 rows of one 16-byte LDS read cover all 64 banks.
__device__ __forceinline__ int gen_swz(int r) { return (r >> 1) & (kGenCH - 1); }

struct GenArgs {
  // first launch
  int64_t nbw;          // weight work-groups
  int row_waves;        // waves per weight row: 1 or 4
  int64_t rows;         // weight rows of all groups
  int64_t icg, taps;    // channels per group and taps of a weight row (Linear: K, 1)
  int a4, hilo, xt, xmode;  // xmode 0: NCHW transpose, 1: rows of channels, 2: in place
  // operands
  uint16_t* wd;
  float* rs;
  uint16_t* xh;
  uint32_t* flags;
  uint32_t* zero;       // 16 zeroed bytes
  float* part;
  int64_t cg, kp, ldw;  // padded channels per group, k of a plane, weight row pitch (planes * kp)
  int64_t pixels, planes, cpl;  // rows of x, flag planes, planes per group
  // GEMM
  const uint16_t* xa;
  uint32_t xpitch;      // halves of a pixel in xa
  uint32_t xgroup;      // halves between groups within a pixel
  int splits;
};

// ---- first launch ------------------------------------------------------------

// Index at bit position `bit` of the packed bytes w: BITS = 3 may straddle
// two bytes, and its second byte then lies inside the stream.
template <int BITS>
__device__ __forceinline__ uint32_t gen_index(const uint8_t* w, int64_t bit) {
  const int64_t b = bit >> 3;
  const int sh = static_cast<int>(bit & 7);
  uint32_t v = w[b];
  if constexpr (BITS == 3) {
    if (sh > 5) v |= static_cast<uint32_t>(w[b + 1]) << 8;
  }
  return (v >> sh) & ((1u << BITS) - 1u);
}

// kGenRows weight rows of one wave each, or one row of all four (a.row_waves).
// Their packed bytes are first copied into LDS with coalesced loads (a 3x3
// row's indices are 8 single bytes per 8 weights: gathered from memory they
// cost more than the GEMM's share of them), the codebook row's scaled fp16
// entries (hi, and lo = what hi leaves of them) into a table per wave; then 8
// weights per lane and trip.  Rows too long for the copy are gathered from
// memory.  512 rows of 4,608 4-bit weights: 13.3 -> 10.8 us.
template <int BITS>
__device__ void gen_weight_rows(const GemmArgs& p, const GenArgs& a, int64_t b) {
  constexpr int E = 1 << BITS;
  __shared__ uint16_t tab[kGenRows][2][E];
  __shared__ __attribute__((aligned(16))) uint8_t raw[kGenRaw + 8];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t row_a = a.row_waves == 4 ? b : b * kGenRows;  // first row of this work-group
  const int64_t nrow = a.row_waves == 4 ? 1 : (a.rows - row_a < kGenRows ? a.rows - row_a : kGenRows);
  const int64_t kw = a.icg * a.taps;  // indices of a packed row
  const int64_t byte0 = row_a * kw * BITS >> 3, byte1 = ((row_a + nrow) * kw * BITS + 7) >> 3;
  const bool staged = byte1 - byte0 <= kGenRaw;
  // byte i of the copy is p.w[org + i]; org keeps whole aligned words where p.w is aligned
  const bool words = (reinterpret_cast<uintptr_t>(p.w) & 3) == 0;
  const int64_t org = words ? byte0 & ~int64_t(3) : byte0;
  if (staged) {
    const int nb = static_cast<int>(byte1 - org), nw = words ? nb >> 2 : 0;
    for (int i = threadIdx.x; i < nw; i += 256)
      reinterpret_cast<uint32_t*>(raw)[i] = reinterpret_cast<const uint32_t*>(p.w + org)[i];
    for (int i = 4 * nw + threadIdx.x; i < nb; i += 256) raw[i] = p.w[org + i];
  }
  const int64_t row = a.row_waves == 4 ? row_a : row_a + wave;
  const int64_t cbrow = p.cb_rows == 1 ? 0 : row < a.rows ? row : a.rows - 1;
  constexpr int EPL = (E + 63) / 64;
  float c[EPL], mx = 0.0f;
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    const int j = lane + 64 * i;
    c[i] = j < p.cb_size ? load_as_float(p.cb, p.cb_dt, cbrow * p.cb_size + j) : 0.0f;
    mx = fmaxf(mx, fabsf(c[i]));
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) mx = fmaxf(mx, __shfl_xor(mx, m, 64));
  const int e = cb_exponent(mx);
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    const int j = lane + 64 * i;
    if (j < E) {
      const float v = ldexpf(c[i], e);
      const uint32_t h = float_to_f16_bits(v);
      tab[wave][0][j] = static_cast<uint16_t>(h);
      tab[wave][1][j] = static_cast<uint16_t>(float_to_f16_bits(v - f16_bits_to_float(h)));
    }
  }
  __syncthreads();
  if (row >= a.rows) return;
  if (lane == 0 && (a.row_waves == 1 || wave == 0)) a.rs[row] = ldexpf(p.acc_scale, -e);
  const uint8_t* src = staged ? raw : p.w;
  const int64_t row0 = row * kw * BITS - (staged ? 8 * org : 0);  // bit of the row's first index in src
  const int64_t chunks = a.kp >> 3;
  const bool bytes = a.taps == 1 && (row0 & 7) == 0;  // a chunk's 8 indices are BITS whole bytes
  uint16_t* out = a.wd + row * a.ldw;
  for (int64_t q = a.row_waves == 4 ? threadIdx.x : lane; q < chunks; q += 64 * a.row_waves) {
    uint32_t ix[8];
    const int tap = a.taps == 1 ? 0 : static_cast<int>(static_cast<uint32_t>(8 * q) / static_cast<uint32_t>(a.cg));
    const int64_t c0 = 8 * q - tap * a.cg;
    const int n = tap >= a.taps || c0 >= a.icg ? 0 : a.icg - c0 < 8 ? static_cast<int>(a.icg - c0) : 8;
    if (bytes && n == 8) {
      uint64_t v = 0;
#pragma unroll
      for (int i = 0; i < BITS; ++i) v |= static_cast<uint64_t>(src[(row0 >> 3) + q * BITS + i]) << (8 * i);
#pragma unroll
      for (int i = 0; i < 8; ++i) ix[i] = static_cast<uint32_t>(v >> (i * BITS)) & ((1u << BITS) - 1u);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)  // conv_kcrs: (channel, tap)
        ix[i] = gen_index<BITS>(src, row0 + (i < n ? (c0 + i) * a.taps + tap : 0) * BITS);
    }
#pragma unroll
    for (int pl = 0; pl < 2; ++pl) {
      if (pl == 1 && !a.hilo) break;
      uint32_t h[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t lo = 2 * i < n ? tab[wave][pl][ix[2 * i]] : 0u;
        const uint32_t hi = 2 * i + 1 < n ? tab[wave][pl][ix[2 * i + 1]] : 0u;
        h[i] = lo | (hi << 16);
      }
      *reinterpret_cast<uint4*>(out + pl * a.kp + 8 * q) = make_uint4(h[0], h[1], h[2], h[3]);
    }
  }
}

// 8 activations (the first `n` of them real) -> fp16 or W4A4 codes.
__device__ __forceinline__ uint4 gen_convert8(const GemmArgs& p, const GenArgs& a, float (&v)[8], int n) {
  if (a.a4) u4_codes<8>(v, p.act_scale, p.act_zp);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = i < n ? v[i] : 0.0f;
  return make_uint4(f16x2_rne(v[0], v[1]), f16x2_rne(v[2], v[3]), f16x2_rne(v[4], v[5]), f16x2_rne(v[6], v[7]));
}

__device__ __forceinline__ int dtype_bytes(int dt) { return dt == DIMQ_F64 ? 8 : dt == DIMQ_F32 ? 4 : 2; }

__device__ __forceinline__ uint32_t gen_big(uint4 h) { return ((h.x | h.y) | (h.z | h.w)) & kRangeBigBits; }

// NCHW -> pixel rows: 64 pixels x 64 channels of one group per work-group.
// Loads run along the pixels of a channel plane, stores along the channels of
// a pixel (128 bytes), so both sides are whole runs.
template <class T, class ToF>
__device__ __forceinline__ void gen_plane_load(const T* __restrict__ x, int64_t at, int64_t hw, int n, ToF f,
                                               float (&v)[8]) {
  T r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = x[at + (i < n ? i : n - 1) * hw];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = f(r[i]);
}

__device__ void gen_transpose(const GemmArgs& p, const GenArgs& a, int64_t b) {
  __shared__ __attribute__((aligned(16))) uint4 tile[kGenPix][kGenChan / 8 + 1];
  // 32-bit divisions: the plan keeps pixels times channels below 2^31
  const uint32_t ptiles = static_cast<uint32_t>((a.pixels + kGenPix - 1) / kGenPix);
  const int64_t plane = static_cast<uint32_t>(b) / ptiles, pt = b - plane * ptiles;
  const int64_t grp = static_cast<uint32_t>(plane) / static_cast<uint32_t>(a.cpl);
  const int64_t cb0 = (plane - grp * a.cpl) * kGenChan;
  const int64_t hw = p.cH * p.cW;
  const int64_t pix = pt * kGenPix + (threadIdx.x & 63);
  const int64_t pixc = pix < a.pixels ? pix : a.pixels - 1;
  const int64_t img = static_cast<uint32_t>(pixc) / static_cast<uint32_t>(hw), r = pixc - img * hw;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int cq = (threadIdx.x >> 6) + 4 * u;
    const int64_t c0 = cb0 + 8 * cq;
    if (c0 >= a.cg) continue;
    const int n = a.icg - c0 < 8 ? static_cast<int>(a.icg - c0) : 8;
    const int64_t at = (img * p.cC + grp * a.icg + c0) * hw + r;
    float v[8];
    switch (a.xt) {
      case DIMQ_F32: gen_plane_load(static_cast<const float*>(p.x), at, hw, n, [](float t) { return t; }, v); break;
      case DIMQ_F16:
        gen_plane_load(static_cast<const uint16_t*>(p.x), at, hw, n, [](uint16_t t) { return f16_bits_to_float(t); }, v);
        break;
      case DIMQ_BF16:
        gen_plane_load(static_cast<const uint16_t*>(p.x), at, hw, n, [](uint16_t t) { return bf16_bits_to_float(t); }, v);
        break;
      default:
        gen_plane_load(static_cast<const double*>(p.x), at, hw, n, [](double t) { return (float)t; }, v);
    }
    tile[threadIdx.x & 63][cq] = gen_convert8(p, a, v, n);
  }
  __syncthreads();
  const int64_t left = (a.cg - cb0) >> 3;  // 16-byte chunks of a pixel in this tile
  const int nq = left < kGenChan / 8 ? static_cast<int>(left) : kGenChan / 8;
  const int q = threadIdx.x & 7;
  for (int t = threadIdx.x >> 3; t < kGenPix; t += 32) {
    const int64_t px = pt * kGenPix + t;
    uint4 h = q < nq ? tile[t][q] : make_uint4(0, 0, 0, 0);
    if (px < a.pixels && q < nq) *reinterpret_cast<uint4*>(a.xh + px * a.xpitch + grp * a.xgroup + cb0 + 8 * q) = h;
    if (a.planes) {
      uint32_t big = gen_big(h);
      big |= __shfl_xor(big, 1, 64);
      big |= __shfl_xor(big, 2, 64);
      big |= __shfl_xor(big, 4, 64);
      if (q == 0 && px < a.pixels) a.flags[plane * a.pixels + px] = big;
    }
  }
}

// Rows of channels (channels-last pixels, or a Linear's activation rows): 64
// channels of one row and group per 8 lanes.
__device__ void gen_rows(const GemmArgs& p, const GenArgs& a, int64_t b) {
  const int64_t per_row = a.cpl * (p.conv ? p.groups : 1);
  const int64_t task = b * 32 + (threadIdx.x >> 3);
  const int q = threadIdx.x & 7;
  const int64_t px = static_cast<uint32_t>(task) / static_cast<uint32_t>(per_row);
  if (px >= a.pixels) return;  // the 8 lanes of a task leave together
  const int64_t plane = task - px * per_row;
  const int64_t grp = static_cast<uint32_t>(plane) / static_cast<uint32_t>(a.cpl);
  const int64_t c0 = (plane - grp * a.cpl) * kGenChan + 8 * q;
  const int64_t left = a.icg - c0;
  const int n = left < 0 ? 0 : left < 8 ? static_cast<int>(left) : 8;
  const int64_t at = px * (p.conv ? p.cC : p.ldx) + grp * a.icg + c0;
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = 0.0f;
  if (n > 0) {
    const bool vec = n == 8 && ((reinterpret_cast<uintptr_t>(p.x) + at * dtype_bytes(a.xt)) & 15) == 0;
    if (vec && a.xt == DIMQ_F32) {
      const float4* s4 = reinterpret_cast<const float4*>(static_cast<const float*>(p.x) + at);
      const float4 u = s4[0], w = s4[1];
      v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w; v[4] = w.x; v[5] = w.y; v[6] = w.z; v[7] = w.w;
    } else if (vec && (a.xt == DIMQ_F16 || a.xt == DIMQ_BF16)) {
      const uint4 u = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(p.x) + at);
      const uint32_t h[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[2 * i] = a.xt == DIMQ_F16 ? f16_bits_to_float(h[i] & 0xffffu) : bf16_bits_to_float(h[i] & 0xffffu);
        v[2 * i + 1] = a.xt == DIMQ_F16 ? f16_bits_to_float(h[i] >> 16) : bf16_bits_to_float(h[i] >> 16);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = load_as_float(p.x, a.xt, at + (i < n ? i : n - 1));
    }
  }
  const uint4 h = gen_convert8(p, a, v, n);
  if (c0 < a.cg) *reinterpret_cast<uint4*>(a.xh + px * a.xpitch + grp * a.xgroup + c0) = h;
  if (a.planes) {
    uint32_t big = gen_big(h);
    big |= __shfl_xor(big, 1, 64);
    big |= __shfl_xor(big, 2, 64);
    big |= __shfl_xor(big, 4, 64);
    if (q == 0) a.flags[plane * a.pixels + px] = big;
  }
}

template <int BITS>
__global__ __launch_bounds__(256) void gen_prep_kernel(const GemmArgs p, const GenArgs a) {
  const int64_t b = blockIdx.x;
  if (b == 0 && threadIdx.x < 4) a.zero[threadIdx.x] = 0u;
  if (b < a.nbw) {
    gen_weight_rows<BITS>(p, a, b);
  } else if (a.xmode == 0) {
    gen_transpose(p, a, b - a.nbw);
  } else {
    gen_rows(p, a, b - a.nbw);
  }
}

// ---- outputs -----------------------------------------------------------------

// Whether some activation that rows [m0, m0 + rows) of group grp read has
// magnitude >= 2^-7 (the range guard's test on its fp16 value, common.h);
// work-group-uniform.  Mostly the first flags looked at say so.
template <bool CONV>
__device__ bool gen_seen_big(const GemmArgs& p, const GenArgs& a, int64_t m0, int rows, int64_t grp) {
  const int r = threadIdx.x;
  const int64_t m = m0 + r;
  const bool mine = r < rows && m < p.M;
  int64_t img = 0;
  int ih0 = 0, iw0 = 0;
  if (CONV && mine) {
    const int64_t hw = p.cOH * p.cOW;
    img = static_cast<uint32_t>(m) / static_cast<uint32_t>(hw);
    const int t = static_cast<int>(m - img * hw), oh = t / static_cast<int>(p.cOW);
    ih0 = oh * p.csh - p.cph;
    iw0 = (t - oh * static_cast<int>(p.cOW)) * p.csw - p.cpw;
  }
  for (int64_t tap = 0; tap < a.taps; ++tap) {
    uint32_t big = 0;
    if (mine) {
      int64_t px = m;
      bool in = true;
      if (CONV) {
        const int kh = static_cast<int>(tap) / p.cKW, kw = static_cast<int>(tap) - kh * p.cKW;
        const int ih = ih0 + kh * p.cdh, iw = iw0 + kw * p.cdw;
        in = ih >= 0 && ih < p.cH && iw >= 0 && iw < p.cW;
        px = (img * p.cH + ih) * p.cW + iw;
      }
      if (in)
        for (int64_t c = 0; c < a.cpl && !big; ++c) big = a.flags[(grp * a.cpl + c) * a.pixels + px];
    }
    if (__syncthreads_or(big != 0u)) return true;
  }
  return false;
}

// ---- the GEMM ------------------------------------------------------------------

// A 64 x 64 tile of y, four waves of 32 x 32 (weights as the MFMA's A operand,
// rows = output columns, activations as B, so a lane's accumulator holds 4
// consecutive columns of one row), 48 KB of LDS: three work-groups per CU.
// SPLIT: the k range blockIdx.y of a.splits, fp32 sums to a.part in y's
// element order.  Tiles of 128 x 64, 64 x 128 and 128 x 128, 32-k stages, four
// to five slots and waves that share a tile along k were all measured at seven
// shapes and nowhere faster by more than a twentieth: these shapes leave the
// chip short of work-groups, or (W4A4 conv2d_lut, 32 x 256 x 14 x 14, 392
// tiles: 24 us; 128 x 128: 46) of waves to hide a stage's latency behind.
template <bool CONV, bool GUARD, bool SPLIT>
__global__ __launch_bounds__(256) void gen_gemm_kernel(const GemmArgs p, const GenArgs a, int bits) {
  constexpr int NT = 256, NW = 4, B = kGenB, S = kGenS;
  constexpr int RB = 16 * kGenCH, RPB = 64 / kGenCH;  // bytes of a stage row, rows of one wave-wide load
  constexpr int RSTAGE = 2 * B * RB;
  constexpr int J = B / RPB / NW;                     // loads per lane, stage and operand
  constexpr int OTP = B + 4;                          // pitch of the epilogue's parked rows
  static_assert(J * RPB * NW == B, "every wave issues the same loads");
  static_assert(B * OTP * 4 + 2 * B * 4 <= S * RSTAGE, "the parked tile and the column factors fit in the ring");
  __shared__ __attribute__((aligned(16))) uint8_t sm[S * RSTAGE];
  float* escale = reinterpret_cast<float*>(sm + S * RSTAGE) - 2 * B;
  float* ebias = escale + B;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 31, g = lane >> 5;
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t grp = blockIdx.z;
  int64_t mt, nt;
  tile_coords((p.N + B - 1) / B, mt, nt);
  const int64_t m0 = mt * B, n0 = nt * B;

  float my_scale = 0.0f, my_bias = 0.0f;
  if (!SPLIT && tid < B) {
    const int64_t n = grp * p.N + (n0 + tid < p.N ? n0 + tid : p.N - 1);
    my_scale = a.rs[n];
    if (p.bias) my_bias = load_as_float(p.bias, p.bias_dt, n);
  }

  // stages [k0, k1) of all
  const int64_t nka = a.kp / kGenK, nkt = a.ldw / kGenK;
  int64_t k0 = 0, k1 = nkt;
  if (SPLIT) {
    k0 = nkt * blockIdx.y / a.splits;
    k1 = nkt * (blockIdx.y + 1) / a.splits;
  }
  // lane l fills LDS chunk l % 8 of row 8 b + l / 8 with global chunk (l % 8)
  // ^ swizzle, the same for all of its rows (b = 4 j + wave); rows past N or M
  // repeat the last one (not stored)
  const int rl = RPB * wave + lane / kGenCH;
  const int cq = (lane % kGenCH) ^ gen_swz(rl);
  const uint16_t* wsrc[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int64_t n = n0 + RPB * NW * j + rl;
    wsrc[j] = a.wd + (grp * p.N + (n < p.N ? n : p.N - 1)) * a.ldw + 8 * cq + k0 * kGenK;
  }
  const uint16_t* xg = a.xa + grp * a.xgroup;
  const uint16_t* xsrc[J];
  int ih0[J], iw0[J];
  uint32_t xoff[J];  // halves of (image, ih0, iw0), modulo 2^32
#pragma unroll
  for (int j = 0; j < J; ++j) {
    int64_t m = m0 + RPB * NW * j + rl;
    m = m < p.M ? m : p.M - 1;
    if constexpr (CONV) {
      const uint32_t hw = static_cast<uint32_t>(p.cOH * p.cOW), mu = static_cast<uint32_t>(m);
      const uint32_t img = mu / hw, t = mu - img * hw, oh = t / static_cast<uint32_t>(p.cOW);
      ih0[j] = static_cast<int>(oh) * p.csh - p.cph;
      iw0[j] = static_cast<int>(t - oh * static_cast<uint32_t>(p.cOW)) * p.csw - p.cpw;
      xoff[j] = (img * static_cast<uint32_t>(p.cH * p.cW) +
                 static_cast<uint32_t>(ih0[j] * static_cast<int>(p.cW) + iw0[j])) * a.xpitch;
    } else {
      xsrc[j] = xg + m * a.xpitch + 8 * cq;
    }
  }
  // this lane's place in its plane's k: stage ka, tap (kh, kw), channel c0
  int64_t ka = k0 % nka;
  const int cg = static_cast<int>(a.cg);
  int kh = 0, kw = 0, c0 = 0;
  auto place = [&](int64_t k) {
    const int tap = static_cast<int>(k / cg);
    c0 = static_cast<int>(k - static_cast<int64_t>(tap) * cg);
    kh = tap / p.cKW;
    kw = tap - kh * p.cKW;
  };
  if constexpr (CONV) place(ka * kGenK + 8 * cq);
  const uint32_t smb = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void_g*)sm));
  // the next stage in order (every stage is issued once, in k order) into ring slot `slot`
  auto issue = [&](int64_t kt, int slot) {
    if (kt >= k1) return;
    const uint32_t dst = smb + slot * RSTAGE + wave * 1024;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      dma16(wsrc[j], dst + j * NW * 1024);
      wsrc[j] += kGenK;
    }
    if constexpr (CONV) {
      const int dh = kh * p.cdh, dw = kw * p.cdw;
      const uint32_t delta = static_cast<uint32_t>(dh * static_cast<int>(p.cW) + dw) * a.xpitch + c0;
      const bool tap_in = kh < p.cKH;
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const bool in = tap_in && static_cast<uint32_t>(ih0[j] + dh) < static_cast<uint32_t>(p.cH) &&
                        static_cast<uint32_t>(iw0[j] + dw) < static_cast<uint32_t>(p.cW);
        const void* src = in ? static_cast<const void*>(xg + (xoff[j] + delta)) : static_cast<const void*>(a.zero);
        dma16(src, dst + (J + j) * NW * 1024);
      }
      if (++ka == nka) {  // the second weight plane starts over
        ka = 0;
        place(8 * cq);
      } else {
        c0 += kGenK;
#pragma unroll 1
        while (c0 >= cg) {
          c0 -= cg;
          if (++kw == p.cKW) kw = 0, ++kh;
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < J; ++j) dma16(xsrc[j] + ka * kGenK, dst + (J + j) * NW * 1024);
      if (++ka == nka) ka = 0;
    }
  };

  floatx16g acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
  const int sw = gen_swz(col);
  half8 wf[2][4], xf[2][4];  // fragments of two consecutive stages, four k16 steps each
  auto load = [&](int slot, auto bufc) {
    constexpr int F = decltype(bufc)::value;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint8_t* base = sm + slot * RSTAGE + col * RB + (((2 * i + g) ^ sw) << 4);
      wf[F][i] = *reinterpret_cast<const half8*>(base + wn * 32 * RB);
      xf[F][i] = *reinterpret_cast<const half8*>(base + (B + wm * 32) * RB);
    }
  };
  auto mma = [&](auto bufc) {
    constexpr int F = decltype(bufc)::value;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = mfma32(wf[F][i], xf[F][i], acc);
  };

  // Ring of S slots, stage kt in slot kt % S.  Stage kt + 1's fragments are
  // read whole, behind the barrier that publishes it and ahead of stage kt's
  // MFMAs: with wave tiles this small a lookahead of one k16 step left the
  // waves waiting for LDS.  The same barrier frees stage kt's slot (its
  // fragments are in registers everywhere) for stage kt + S.  No branch lies
  // between a stage's reads and its MFMAs (the compiler would wait for the
  // reads at the join).
  constexpr int LPS = 2 * J;  // loads per lane and stage
  const int64_t nk = k1 - k0;
#pragma unroll
  for (int s = 0; s < S; ++s) issue(k0 + s, s);
  if (nk >= S) wait_vmcnt<(S - 1) * LPS>();
  else wait_vmcnt<0>();
  lds_barrier();
  load(0, std::integral_constant<int, 0>());
  int slot = 0;
  auto step = [&](int64_t kt, auto curc) {  // kt + 1 < nk
    constexpr int CUR = decltype(curc)::value;
    const int next = slot == S - 1 ? 0 : slot + 1;
    if (kt + S <= nk) wait_vmcnt<(S - 2) * LPS>();  // stages kt + 2 .. kt + S - 1 may be in flight
    else wait_vmcnt<0>();
    lds_barrier();
    issue(k0 + kt + S, slot);
    load(next, std::integral_constant<int, 1 - CUR>());
    mma(curc);
    slot = next;
  };
  int64_t kt = 0;
  for (; kt + 2 < nk; kt += 2) {
    step(kt, std::integral_constant<int, 0>());
    step(kt + 1, std::integral_constant<int, 1>());
  }
  if (kt + 1 < nk) {
    step(kt, std::integral_constant<int, 0>());
    mma(std::integral_constant<int, 1>());
  } else {
    mma(std::integral_constant<int, 0>());
  }
  __syncthreads();  // every wave is done with the ring before it is reused
  if constexpr (GUARD) {
    const bool seen = gen_seen_big<CONV>(p, a, m0, B, grp);
    if constexpr (SPLIT) {  // NaN partial outputs: the second pass recomputes what they reach
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[i] = seen ? acc[i] : __builtin_nanf("");
    } else {
      const int bad = __syncthreads_or(!finite_acc<1>(&acc, 1, 1));
      if (bad || !seen) {
        exact_tile_out(p, a.xt, bits, m0, m0 + B, n0, n0 + B, grp);
        return;
      }
    }
  }
  if (!SPLIT && tid < B) {
    escale[tid] = my_scale;
    ebias[tid] = my_bias;
  }
  // The tile, parked as fp32 rows, leaves as 8 columns of a row per thread
  // where y is row-major in whole 16-byte pieces; otherwise one element per
  // thread, the lanes along y's contiguous direction (columns, or for NCHW
  // the pixels).
  float* ot = reinterpret_cast<float*>(sm);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    *reinterpret_cast<float4*>(ot + (wm * 32 + col) * OTP + wn * 32 + 8 * j + 4 * g) =
        make_float4(acc[4 * j], acc[4 * j + 1], acc[4 * j + 2], acc[4 * j + 3]);
  __syncthreads();
  const bool nchw = CONV && p.y_layout == DIMQ_NCHW;
  const int64_t ldy = CONV ? p.cOC : p.ldy;
  const int64_t total = p.M * ldy;  // elements of y (and of one partial plane)
  void* yb = SPLIT ? static_cast<void*>(a.part + blockIdx.y * total) : p.y;
  const int ydt = SPLIT ? static_cast<int>(DIMQ_F32) : p.y_dt;
  const bool vec8 = !nchw && ldy % 8 == 0 && (grp * p.N) % 8 == 0 && (reinterpret_cast<uintptr_t>(yb) & 15) == 0;
  if (vec8) {
    const int q = 8 * (tid & 7);
    const int64_t n = n0 + q;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int r = (tid >> 3) + 32 * u;
      const int64_t m = m0 + r;
      if (m >= p.M || n >= p.N) continue;
      const int64_t off = m * ldy + grp * p.N + n;
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[i] = ot[r * OTP + q + i];
        if constexpr (!SPLIT) v[i] = v[i] * escale[q + i] + ebias[q + i];
      }
      if (n + 8 <= p.N) {
        if constexpr (!SPLIT) epiN<8>(p.epi, off, v, true);
        if (ydt == DIMQ_F32) {
          float* yp = static_cast<float*>(yb) + off;
          *reinterpret_cast<float4*>(yp) = make_float4(v[0], v[1], v[2], v[3]);
          *reinterpret_cast<float4*>(yp + 4) = make_float4(v[4], v[5], v[6], v[7]);
        } else {
          uint32_t h[4];
#pragma unroll
          for (int i = 0; i < 4; ++i)
            h[i] = ydt == DIMQ_F16 ? f16x2_rne(v[2 * i], v[2 * i + 1]) : bf16x2_rne(v[2 * i], v[2 * i + 1]);
          *reinterpret_cast<uint4*>(static_cast<uint16_t*>(yb) + off) = make_uint4(h[0], h[1], h[2], h[3]);
        }
      } else {
        for (int i = 0; i < 8; ++i)
          if (n + i < p.N) store_from_float(yb, ydt, off + i, SPLIT ? v[i] : epi1(p.epi, off + i, v[i]));
      }
    }
  } else {
    const int fast = tid & 63, slow = tid >> 6;
    const int64_t yrow = nchw && m0 + fast < p.M ? out_offset(p, m0 + fast, 0) : 0;
    const int64_t cstep = p.cOH * p.cOW;
#pragma unroll 4
    for (int u = 0; u < B * B / NT; ++u) {
      const int r = nchw ? fast : slow + 4 * u, c = nchw ? slow + 4 * u : fast;
      const int64_t m = m0 + r, n = n0 + c;
      if (m >= p.M || n >= p.N) continue;
      const int64_t off = nchw ? yrow + (grp * p.N + n) * cstep : m * ldy + grp * p.N + n;
      float v = ot[r * OTP + c];
      if constexpr (!SPLIT) v = epi1(p.epi, off, v * escale[c] + ebias[c]);
      store_from_float(yb, ydt, off, v);
    }
  }
}

// Adds the partial outputs of a tile's k ranges in order, then the column
// factors (rs, null: the partial outputs have them), bias and epilogue.  Tiles
// of 16 rows x 64 columns (NCHW: 64 x 16, the lanes along y's contiguous
// direction), four outputs per thread, so that small outputs still make many
// work-groups.  GUARD (fp32 / bf16 activations): a sum that is not finite --
// an activation beyond fp16's range, or the NaN that a tile without any large
// activation writes -- has the tile recomputed in fp32.
template <bool GUARD>
__global__ __launch_bounds__(256) void split_reduce_kernel(const GemmArgs p, const float* __restrict__ part, int splits,
                                                           const float* __restrict__ rs, int xt, int bits,
                                                           bool tapmajor) {
  constexpr int U = 4;
  const bool nchw = p.conv && p.y_layout == DIMQ_NCHW;
  const int tm = nchw ? 64 : 16, tn = nchw ? 16 : 64;
  const int64_t ntn = (p.N + tn - 1) / tn;
  const int64_t mt = blockIdx.x / ntn, m0 = mt * tm, n0 = (blockIdx.x - mt * ntn) * tn, grp = blockIdx.z;
  const int64_t ldy = p.conv ? p.cOC : p.ldy, total = p.M * ldy, cstep = p.cOH * p.cOW;
  const int fast = threadIdx.x & 63, slow = threadIdx.x >> 6;
  int64_t offs[U];
  float v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {  // outputs past M or N re-read the tile's first
    int64_t m = m0 + (nchw ? fast : slow + 4 * u), n = n0 + (nchw ? slow + 4 * u : fast);
    m = m < p.M ? m : m0;
    n = n < p.N ? n : n0;
    offs[u] = nchw ? out_offset(p, m, 0) + (grp * p.N + n) * cstep : m * ldy + grp * p.N + n;
    v[u] = 0.0f;
  }
  // one plane at a time: with every plane's loads in flight at once, whose
  // addresses differ by a multiple of a plane's size, the pass takes up to twice
  // as long (8 planes of 3,136 x 256: 10.7 us against 6)
#pragma unroll 1
  for (int k = 0; k < splits; ++k)
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] += part[k * total + offs[u]];
  if constexpr (GUARD) {
    bool finite = true;
#pragma unroll
    for (int u = 0; u < U; ++u) finite &= __builtin_isfinite(v[u]);
    if (__syncthreads_or(!finite)) {
      exact_tile_out(p, xt, bits, m0, m0 + tm, n0, n0 + tn, grp, tapmajor);
      return;
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t m = m0 + (nchw ? fast : slow + 4 * u), n = n0 + (nchw ? slow + 4 * u : fast);
    if (m >= p.M || n >= p.N) continue;
    const int64_t ng = grp * p.N + n;
    const float b = p.bias ? load_as_float(p.bias, p.bias_dt, ng) : 0.0f;
    store_from_float(p.y, p.y_dt, offs[u], epi1(p.epi, offs[u], v[u] * (rs ? rs[ng] : 1.0f) + b));
  }
}

// ---- host ----------------------------------------------------------------------

int64_t up256(int64_t b) { return (b + 255) / 256 * 256; }
int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

template <bool CONV, bool GUARD>
void launch_gen_gemm(const GemmArgs& p, const GenArgs& a, int bits, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(cdiv(p.M, kGenB) * cdiv(p.N, kGenB)), static_cast<unsigned>(a.splits),
                  static_cast<unsigned>(CONV ? p.groups : 1));
  if (a.splits > 1) {
    hipLaunchKernelGGL((gen_gemm_kernel<CONV, GUARD, true>), grid, dim3(256), 0, s, p, a, bits);
    launch_split_reduce(p, a.part, a.splits, a.rs, a.xt, bits, GUARD, false, s);
  } else {
    hipLaunchKernelGGL((gen_gemm_kernel<CONV, GUARD, false>), grid, dim3(256), 0, s, p, a, bits);
  }
}

}  // namespace

int split_ranges(int64_t tiles, int64_t stages, double us_per_stage, int64_t outputs) {
  const double cus = device_cus();
  double best = 0.0;
  int pick = 1;
  for (int sp = 1; sp <= 8 && sp <= stages / 2; ++sp) {
    const double full = tiles * sp / cus;  // work-groups per CU
    const double us = static_cast<double>(stages) / sp * us_per_stage * (full > 1.0 ? full : 1.0) +
                      (sp > 1 ? 5.0 + 2e-6 * sp * outputs : 0.0);
    if (sp == 1 || us < 0.9 * best) best = us, pick = sp;
  }
  return pick;
}

void launch_split_reduce(const GemmArgs& p, const float* part, int splits, const float* rs, int x_dtype, int bits,
                         bool guard, bool tapmajor, hipStream_t s) {
  const int64_t tm = p.conv && p.y_layout == DIMQ_NCHW ? 64 : 16, tn = 80 - tm;
  const dim3 grid(static_cast<unsigned>(cdiv(p.M, tm) * cdiv(p.N, tn)), 1,
                  static_cast<unsigned>(p.conv ? p.groups : 1));
  if (guard)
    hipLaunchKernelGGL(split_reduce_kernel<true>, grid, dim3(256), 0, s, p, part, splits, rs, x_dtype, bits, tapmajor);
  else
    hipLaunchKernelGGL(split_reduce_kernel<false>, grid, dim3(256), 0, s, p, part, splits, rs, x_dtype, bits, tapmajor);
}

GenPlan gen_plan(const GemmArgs& p, int bits, int x_dtype, bool a4, bool in_place) {
  GenPlan g;
  if (!(bits == 2 || bits == 3 || bits == 4 || bits == 8) || (a4 && bits != 4)) return g;
  if (!(x_dtype == DIMQ_F16 || x_dtype == DIMQ_BF16 || x_dtype == DIMQ_F32 || (a4 && x_dtype == DIMQ_F64))) return g;
  if (p.M <= 0 || p.N <= 0 || p.K <= 0) return g;
  g.conv = p.conv != 0;
  g.a4 = a4;
  g.hilo = a4 && p.cb_dt != DIMQ_F16;  // fp16 entries are exact in one plane
  const int64_t groups = g.conv ? p.groups : 1, taps = g.conv ? static_cast<int64_t>(p.cKH) * p.cKW : 1;
  const int64_t icg = g.conv ? p.cICg : p.K;
  g.pixels = g.conv ? p.cB * p.cH * p.cW : p.M;
  g.direct_x = in_place && !a4 && x_dtype == DIMQ_F16 &&
               (g.conv ? p.x_layout == DIMQ_NHWC && icg % 8 == 0 : p.K % kGenK == 0 && p.ldx % 8 == 0);
  g.cg = g.conv ? (icg + 7) / 8 * 8 : cdiv(icg, kGenK) * kGenK;
  g.kp = cdiv(taps * g.cg, kGenK) * kGenK;
  const int64_t xpitch = g.direct_x ? (g.conv ? p.cC : p.ldx) : groups * g.cg;
  // 32-bit pixel offsets and row numbers in the kernel
  if (g.pixels * xpitch >= (1ll << 31) || p.M >= (1ll << 31) - 256 || p.N >= (1ll << 31) - 256) return g;
  if (g.conv && (p.cH * p.cW >= (1ll << 31) || taps * g.cg >= (1ll << 30))) return g;
  // a launch dimension holds fewer than 2^32 threads; the tiles without a workspace are larger
  if (cdiv(p.M, kGenB) * cdiv(p.N, kGenB) >= (1ll << 24)) return g;
  const int64_t rows = groups * p.N, ldw = g.kp * (g.hilo ? 2 : 1), nk = ldw / kGenK;
  const int64_t cpl = cdiv(g.cg, kGenChan);
  const bool guard = !a4 && (x_dtype == DIMQ_F32 || x_dtype == DIMQ_BF16);
  g.planes = guard ? groups * cpl : 0;
  const int64_t units = g.conv ? p.cB : p.M;  // images, or rows
  const int64_t unit_bytes = g.pixels / units * ((g.direct_x ? 0 : xpitch * 2) + g.planes * 4);
  g.step = units;
  if (units * unit_bytes > kGenActBytes) {
    const int64_t most = unit_bytes < kGenActBytes ? kGenActBytes / unit_bytes : 1;
    g.step = cdiv(units, cdiv(units, most));  // passes of about the same size
    if (!g.conv && most >= kGenB) {  // whole tiles of rows
      const int64_t up = cdiv(g.step, kGenB) * kGenB;
      g.step = up <= most ? up : most / kGenB * kGenB;
    }
    g.pixels = g.pixels / units * g.step;
  }
  const int64_t M = p.M / units * g.step;  // rows of a pass
  // a 64-k stage takes about 0.3 us on a CU of its own
  g.splits = split_ranges(cdiv(M, kGenB) * cdiv(p.N, kGenB) * groups, nk, 0.3, M * p.N * groups);
  int64_t at = up256(rows * ldw * 2);
  g.off_rs = at;
  at += up256(rows * 4);
  g.off_zero = at;
  at += 256;
  if (!g.direct_x) {
    g.off_x = at;
    at += up256(g.pixels * xpitch * 2);
  }
  if (g.planes) {
    g.off_flags = at;
    at += up256(g.planes * g.pixels * 4);
  }
  if (g.splits > 1) {
    g.off_part = at;
    at += up256(static_cast<int64_t>(g.splits) * M * (g.conv ? p.cOC : p.ldy) * 4);
  }
  g.bytes = at;
  g.ok = true;
  return g;
}

int launch_gen(const GemmArgs& p, const GenPlan& g, int bits, int x_dtype, void* ws, hipStream_t s) {
  uint8_t* base = static_cast<uint8_t*>(ws);
  const int64_t groups = g.conv ? p.groups : 1;
  GenArgs a{};
  a.rows = groups * p.N;
  a.row_waves = g.kp >= 2048 ? 4 : 1;  // a long row keeps a whole work-group busy
  a.nbw = a.row_waves == 4 ? a.rows : cdiv(a.rows, kGenRows);
  a.taps = g.conv ? static_cast<int64_t>(p.cKH) * p.cKW : 1;
  a.icg = g.conv ? p.cICg : p.K;
  a.a4 = g.a4;
  a.hilo = g.hilo;
  a.xt = x_dtype;
  a.xmode = g.direct_x ? 2 : (g.conv && p.x_layout == DIMQ_NCHW) ? 0 : 1;
  a.wd = reinterpret_cast<uint16_t*>(base);
  a.rs = reinterpret_cast<float*>(base + g.off_rs);
  a.zero = reinterpret_cast<uint32_t*>(base + g.off_zero);
  a.xh = reinterpret_cast<uint16_t*>(base + g.off_x);
  a.flags = reinterpret_cast<uint32_t*>(base + g.off_flags);
  a.part = reinterpret_cast<float*>(base + g.off_part);
  a.cg = g.cg;
  a.kp = g.kp;
  a.ldw = g.kp * (g.hilo ? 2 : 1);
  a.planes = g.planes;
  a.cpl = cdiv(g.cg, kGenChan);
  a.xpitch = static_cast<uint32_t>(g.direct_x ? (g.conv ? p.cC : p.ldx) : groups * g.cg);
  a.xgroup = static_cast<uint32_t>(g.direct_x ? a.icg : g.cg);
  a.splits = g.splits;
  const int64_t units = g.conv ? p.cB : p.M;
  const int64_t unit_m = p.M / units, unit_pixels = g.pixels / g.step;
  const int64_t unit_x = g.conv ? p.cC * p.cH * p.cW : p.ldx, unit_y = unit_m * (g.conv ? p.cOC : p.ldy);
  for (int64_t u = 0; u < units; u += g.step) {
    const int64_t n = units - u < g.step ? units - u : g.step;
    GemmArgs q = p;  // this pass's images: x, y and the residual all have them outermost
    q.x = static_cast<const uint8_t*>(p.x) + u * unit_x * dtype_size(x_dtype);
    q.y = static_cast<uint8_t*>(p.y) + u * unit_y * dtype_size(p.y_dt);
    if (p.epi.res) {
      q.epi.res = static_cast<const uint8_t*>(p.epi.res) + u * unit_y * dtype_size(p.epi.res_dt);
      q.epi.res_vec = aligned(q.epi.res, 16);
    }
    q.M = n * unit_m;
    if (g.conv) q.cB = n;
    a.pixels = n * unit_pixels;
    a.xa = g.direct_x ? static_cast<const uint16_t*>(q.x) : a.xh;
    if (u > 0) a.nbw = 0;  // the weights are laid out
    int64_t nbx = 0;
    if (a.xmode == 0) nbx = cdiv(a.pixels, kGenPix) * groups * a.cpl;
    if (a.xmode == 1) nbx = cdiv(a.pixels * groups * a.cpl, 32);
    const dim3 grid(static_cast<unsigned>(a.nbw + nbx));
    switch (bits) {
      case 2: hipLaunchKernelGGL(gen_prep_kernel<2>, grid, dim3(256), 0, s, q, a); break;
      case 3: hipLaunchKernelGGL(gen_prep_kernel<3>, grid, dim3(256), 0, s, q, a); break;
      case 4: hipLaunchKernelGGL(gen_prep_kernel<4>, grid, dim3(256), 0, s, q, a); break;
      default: hipLaunchKernelGGL(gen_prep_kernel<8>, grid, dim3(256), 0, s, q, a); break;
    }
    const int rc = check_launch("codebook layer (operand layout)");
    if (rc != DIMQ_OK) return rc;
    if (g.conv) {
      if (g.planes) launch_gen_gemm<true, true>(q, a, bits, s);
      else launch_gen_gemm<true, false>(q, a, bits, s);
    } else {
      if (g.planes) launch_gen_gemm<false, true>(q, a, bits, s);
      else launch_gen_gemm<false, false>(q, a, bits, s);
    }
  }
  return check_launch("codebook layer");
}

}  // namespace dimq
