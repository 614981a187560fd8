// Host side of the codebook Linear: argument checks (with the reference's
// messages where one exists, csrc/dimq_gemm_lut.cu:66-79), tile selection and
// launch.
#include <mutex>

#include "gemm_big.h"
#include "gemm_gen.h"
#include "gemm_kernel.h"
#include "gemv_fast.h"

namespace dimq {
namespace {

constexpr int64_t kCUs = 256;

}  // namespace

// gemm_pd.hip: the pre-decoded-weight path for large M (weights decoded once
// per call into the workspace, then an fp16 GEMM fed by global_load_lds).
int64_t predecoded_ws_bytes(int64_t M, int64_t K, int64_t N, int bits, int x_dtype);
int launch_predecoded(const GemmArgs& p, int bits, int x_dtype, void* ws, int64_t ws_bytes, hipStream_t s,
                      const void* decoded = nullptr);
int64_t predecoded_w_bytes(int64_t N, int64_t K, int bits);
int launch_predecode_jobs(const DimqPredecodeJob* jobs, int count, hipStream_t s);

// Fast-path tiles need K % 128 == 0, aligned rows/streams and a Linear layout.
int gemm_fast_tile(int tile, const GemmArgs& p, int bits) {
  if (bits == 8 || p.conv || !p.fast_b || !p.vec_a || p.K % kKM != 0) return tile;
  if (tile == kTile128x64) return kTileFast128x64;
  if (tile == kTile64x32) return kTileFast64x32;
  return tile;
}

// Large-tile kernels (gemm_big.h) for Linear shapes with M > 64, K % 64 == 0
// and aligned rows/streams: tile ids of launch_big_linear_modes, -1 when the
// shape does not qualify.
int gemm_big_tile(const GemmArgs& p, int bits, int x_dtype, int variant) {
  if (variant == DIMQ_VARIANT_SMALL_M || p.conv || !(bits == 2 || bits == 3 || bits == 4)) return -1;
  const int mode = epi_mode(p.epi);  // epilogues the large tiles are instantiated for
  const bool qmode = x_dtype == DIMQ_F16 && (mode == kEpiQuant || mode == (kEpiRelu | kEpiQuant) ||
                                             mode == (kEpiGelu | kEpiQuant));
  if (!(mode == kEpiNone || mode == kEpiRelu || mode == kEpiGelu || mode == kEpiRes || qmode)) return -1;
  if (p.M <= 64 || p.K % 64 != 0 || !p.fast_b || !p.vec_a) return -1;
  // 256x256 shared-decode tiles for large M (measured on the ViT-B/16 shapes at
  // M 12,608, bf16: qkv 84 vs 104 us, proj 40 vs 50, fc1 114 vs 134, fc2 104 vs
  // 133 against the best 128x128 tile); fp32 activations spill its registers.
  if (p.M >= 2048) return x_dtype != DIMQ_F32 ? 10 : p.K >= 2048 ? 2 : 7;
  // Below 2,048 rows the deep-pipeline tile (7, 64x128) is faster than the
  // 128x128 one (2) unless that one's work-groups fill their last round on the
  // CUs (128x128 against 64x128 tiles: M 100, N = K = 4,096, 62 and 45 us; M
  // 500 61 and 41; M 1,576, N 768, K 3,072 47 and 31).  There, 4-bit codebooks
  // on fp16 and fp32 aside, its lower decode work per product wins: N 4,096, K
  // 4,096, M 1,576 (416 tiles) bf16 3-bit 96 and 104 us, fp16 2-bit 73 and 81;
  // M 2,047 (512) 104 and 118, 83 and 90; N 6,144, M 1,300 (528) 138 and 107,
  // 1,800 (720) 151 and 165.  2-bit codes on 16-bit activations, the cheapest
  // to decode, gain from a quarter of a round on (576 and 624 tiles 1.01 to
  // 1.06 times as fast, the other types 0.85 to 1.0).
  if (p.K >= 2048 && (bits < 4 || x_dtype == DIMQ_BF16)) {
    const int64_t tiles = ((p.M + 127) / 128) * ((p.N + 127) / 128), last = tiles % device_cus();
    const bool half = x_dtype != DIMQ_F32;
    if (last == 0 ? tiles > 400 || half : tiles > 400 && last > (bits == 2 && half ? 48 : 150)) return 2;
  }
  return 7;
}

// Whether the general pre-laid path (gemm_gen.hip) takes a Linear that no path
// with a workspace of its own does: every shape beyond the decode shapes that
// the large tiles' k steps or codebooks do not fit.  At 16 < M <= 64 with
// K % 128 == 0 the register-codebook tiles decode each weight once or twice
// only, in a time that hardly depends on N, while laying the weights out grows
// with N.  The general path wins while K is long and N small, up to 2,048
// outputs (2-bit codes, which decode faster, 1,536), from 49 rows on half as
// many more: K 2,048, 4-bit, M 17, N 2,048 22.4 against 20.4 us, N 3,072 22.5
// and 24.8, N 4,096 22.5 and 29.8; M 64, N 3,072 27.0 and 25.3; 2-bit, K 1,536,
// M 17, N 1,536 15.7 and 15.6, N 2,048 15.7 and 16.5; M 32, K 3,072, N 768 31.1
// and 16.8; M 17, K 384, N 3,072 11.7 and 12.2.  W4A4 (a4), whose tiles need
// the activations quantized first: up to 3,072 (K 2,048, M 17, N 3,072 24.0 and
// 23.5, N 4,096 24.2 and 28.4).
// K % 32 == 0 off the large tiles' 64-k steps: the register-codebook tiles'
// 64x128 form, taken below 256 tiles of 128x256, is faster once its tiles fill
// the chip: per k about 23 ns against 0.9 per 1,000 outputs of layout and 4.5
// per million products of M * N here, which is N (M + 200) about 4.8M (W4A4,
// whose activations are quantized first: 5.5M).  N 4,096, K 4,000, M 500 91
// against 57 us, M 1,500 103 and 130, M 2,047 (the other form) 339 and 167; N
// 8,192, K 8,160, M 500 158 and 189.
bool gen_wants_linear(int64_t M, int64_t K, int64_t N, int bits, bool a4 = false) {
  if (M <= 16) return false;
  if (bits == 8) return true;
  if (K % 64 != 0) {
    const bool filled = K % 32 == 0 && K >= 960 && N * (M + 200) > (a4 ? 5500000 : 4800000);
    return !(filled && ((M + 127) / 128) * ((N + 255) / 256) < kCUs);
  }
  if (M > 64) return false;
  if (K % 128 != 0) return true;
  const int64_t most = a4 ? 3072 : bits == 2 ? (M > 48 ? 2048 : 1536) : (M > 48 ? 3072 : 2048);
  return K >= 1024 && N <= most && N * K <= (8ll << 20);
}

// k ranges of a Linear on the 64x128 tiles.  A 64-k stage takes 0.45 us there.
// M 197, N 768, K 3,072 (24 tiles): 29.3 -> 16.2 us in 6 ranges; M 788: 29.6 ->
// 21.3 in 3; M 100, N = K = 4,096: 45.1 -> 22.5 in 4.  At K < 2,048 the second
// launch costs what the ranges save (M 197, N = K = 768: 12.9 against 12.2 to
// 14.0), and at M 500, N = K = 4,096 the tiles fill the chip (41.4, 41.0).
int big_linear_splits(int64_t M, int64_t K, int64_t N, int tile) {
  if (tile != 7 || K < 2048) return 1;
  return split_ranges(((M + 63) / 64) * ((N + 127) / 128), K / 64, 0.45, M * N);
}

int gemm_pick_tile(int64_t M, int64_t N, int variant) {
  if (variant == DIMQ_VARIANT_SMALL_M) return M <= 16 ? kTileGemv : kTile16x16;
  if (variant == DIMQ_VARIANT_AUTO && M <= 16) return kTileGemv;
  const int64_t big = ((M + 127) / 128) * ((N + 255) / 256);
  if (big >= kCUs) return kTile128x64;
  return kTile64x32;
}

namespace {

template <bool A4>
int dispatch(const GemmArgs& p, int bits, int xt, int tile, hipStream_t s) {
#define DIMQ_XT_CASES(B)                                                   \
  switch (xt) {                                                            \
    case DIMQ_F32: return launch_gemm_tile<B, DIMQ_F32, A4>(p, tile, s);   \
    case DIMQ_F16: return launch_gemm_tile<B, DIMQ_F16, A4>(p, tile, s);   \
    case DIMQ_BF16: return launch_gemm_tile<B, DIMQ_BF16, A4>(p, tile, s); \
  }                                                                        \
  break;
  if constexpr (A4) {
    switch (xt) {
      case DIMQ_F32: return launch_gemm_tile<4, DIMQ_F32, true>(p, tile, s);
      case DIMQ_F16: return launch_gemm_tile<4, DIMQ_F16, true>(p, tile, s);
      case DIMQ_BF16: return launch_gemm_tile<4, DIMQ_BF16, true>(p, tile, s);
      case DIMQ_F64: return launch_gemm_tile<4, DIMQ_F64, true>(p, tile, s);
    }
  } else {
    switch (bits) {
      case 2: DIMQ_XT_CASES(2)
      case 3: DIMQ_XT_CASES(3)
      case 4: DIMQ_XT_CASES(4)
      case 8: DIMQ_XT_CASES(8)
    }
  }
#undef DIMQ_XT_CASES
  return set_error(DIMQ_ERR_UNSUPPORTED, "unsupported dtype/bit-width combination (x dtype %d, bits %d)", xt, bits);
}

}  // namespace

int gemm_dispatch(const GemmArgs& p, int bits, int xt, bool a4, int tile, hipStream_t s) {
  return a4 ? dispatch<true>(p, bits, xt, tile, s) : dispatch<false>(p, bits, xt, tile, s);
}

int linear_codebook_impl(const void* x, int x_dtype, int64_t M, int64_t K, int64_t ldx, const uint8_t* packed_w,
                         int bits, const void* codebook, int cb_dtype, int64_t cb_rows, int64_t cb_size,
                         const void* bias, int bias_dtype, int64_t N, void* y, int y_dtype, int64_t ldy,
                         const Epi& epi, int variant, hipStream_t s, float acc_scale = 1.0f,
                         void* workspace = nullptr, int64_t workspace_bytes = 0, const void* decoded = nullptr) {
  GemmArgs p{};
  p.epi = epi;
  p.acc_scale = acc_scale;
  p.x = x;
  p.M = M;
  p.K = K;
  p.ldx = ldx;
  p.w = packed_w;
  p.N = N;
  p.cb = codebook;
  p.cb_dt = cb_dtype;
  p.cb_rows = cb_rows;
  p.cb_size = static_cast<int>(cb_size);
  p.bias = bias;
  p.bias_dt = bias_dtype;
  p.y = y;
  p.y_dt = y_dtype;
  p.ldy = ldy;
  p.act_scale = 1.0f;
  p.act_zp = 0;
  p.fast_b = (K % 32 == 0) && aligned(packed_w, 16);
  const int xs = dtype_size(x_dtype);
  p.vec_a = aligned(x, 16) && ((ldx * xs) % 16 == 0);
  p.groups = 1;
  if (M == 0 || N == 0) return DIMQ_OK;
  if ((workspace != nullptr || decoded != nullptr) && variant != DIMQ_VARIANT_SMALL_M) {
    const int rc = launch_predecoded(p, bits, x_dtype, workspace, workspace_bytes, s, decoded);
    if (rc >= 0) return rc;
  }
  const int big = gemm_big_tile(p, bits, x_dtype, variant);
  if (workspace != nullptr && aligned(workspace, 256)) {
    // the first pass of split k has no epilogue: any may follow in the second
    GemmArgs plain = p;
    plain.epi = Epi{};
    const int tile = gemm_big_tile(plain, bits, x_dtype, variant);
    const int sp = tile >= 0 ? big_linear_splits(M, K, N, tile) : 1;
    if (sp > 1 && workspace_bytes >= split_bytes(sp, M, ldy)) {
      const GemmArgs q = split_args(p, sp, workspace);
      int rc = DIMQ_OK;
      switch (bits) {
        case 2: rc = launch_big_b2(q, x_dtype, tile, s); break;
        case 3: rc = launch_big_b3(q, x_dtype, tile, s); break;
        default: rc = launch_big_b4(q, x_dtype, tile, s); break;
      }
      if (rc != DIMQ_OK) return rc;
      launch_split_reduce(p, static_cast<const float*>(workspace), sp, nullptr, x_dtype, bits, x_dtype != DIMQ_F16,
                          false, s);
      return check_launch("linear_codebook (split k)");
    }
    if (big < 0 && gen_wants_linear(M, K, N, bits) && variant != DIMQ_VARIANT_SMALL_M) {
      const GenPlan g = gen_plan(p, bits, x_dtype, false, aligned(x, 16));
      if (g.ok && workspace_bytes >= g.bytes) return launch_gen(p, g, bits, x_dtype, workspace, s);
    }
  }
  if (big >= 0) {
    switch (bits) {
      case 2: return launch_big_b2(p, x_dtype, big, s);
      case 3: return launch_big_b3(p, x_dtype, big, s);
      default: return launch_big_b4(p, x_dtype, big, s);
    }
  }
  int tile = gemm_fast_tile(gemm_pick_tile(M, N, variant), p, bits);
  if (tile < 0 || tile >= kTileCount) tile = gemm_pick_tile(M, N, variant);
  if (tile >= kTileFast128x64 && gemm_fast_tile(kTile64x32, p, bits) == kTile64x32) tile = gemm_pick_tile(M, N, variant);
  if (tile == kTileGemv && (M > 16 || bits == 8)) tile = gemm_pick_tile(M, N, DIMQ_VARIANT_MFMA);
  // 8-bit: 16-row tiles when the 64-row ones would leave most CUs idle
  // (ResNet-18 fc, M 128 x N 1000: 32 work-groups on 64-row tiles, 128 on
  // 16-row tiles; measured 28.9 -> 23.4 us per call)
  if (bits == 8 && tile == kTile64x32 && ((M + 63) / 64) * ((N + 63) / 64) < kCUs / 2) tile = kTile16x16;
  if (tile == kTileGemv && gemv_direct_ok(p, bits, x_dtype)) {
    switch (bits) {
      case 2: return launch_gemv_direct<2>(p, s);
      case 3: return launch_gemv_direct<3>(p, s);
      default: return launch_gemv_direct<4>(p, s);
    }
  }
  if (tile == kTileGemv) {
    const bool ws_ok = workspace != nullptr && aligned(workspace, 16);
    GemvPlan pl;
    bool planned = gemv_plan(p, bits, ws_ok, pl);
    if (planned && gemv_partial_bytes(p, pl) > (ws_ok ? workspace_bytes : 0)) planned = gemv_plan(p, bits, false, pl);
    if (planned) {
      float* part = static_cast<float*>(workspace);
      switch (bits) {
        case 2: return launch_gemv_stream<2>(p, x_dtype, pl, part, s);
        case 3: return launch_gemv_stream<3>(p, x_dtype, pl, part, s);
        default: return launch_gemv_stream<4>(p, x_dtype, pl, part, s);
      }
    }
  }
  return dispatch<false>(p, bits, x_dtype, tile, s);
}

}  // namespace dimq

using namespace dimq;

static int linear_codebook_checked(const void* x, int x_dtype, int64_t M, int64_t K, const uint8_t* packed_w,
                                   int64_t packed_numel, int bits, const void* codebook, int cb_dtype, int64_t cb_rows,
                                   int64_t cb_size, const void* bias, int bias_dtype, int64_t N, void* y, int y_dtype,
                                   const void* residual, int residual_dtype, int activation, int variant, void* stream,
                                   void* workspace, int64_t workspace_bytes, const void* decoded = nullptr);

extern "C" int dimq_linear_codebook(const void* x, int x_dtype, int64_t M, int64_t K, const uint8_t* packed_w,
                                    int64_t packed_numel, int bits, const void* codebook, int cb_dtype,
                                    int64_t cb_rows, int64_t cb_size, const void* bias, int bias_dtype, int64_t N,
                                    void* y, int y_dtype, int variant, void* stream) {
  return dimq_linear_codebook_ex(x, x_dtype, M, K, packed_w, packed_numel, bits, codebook, cb_dtype, cb_rows, cb_size,
                                 bias, bias_dtype, N, y, y_dtype, nullptr, 0, DIMQ_ACT_NONE, variant, stream);
}

// Workspace of dimq_linear_codebook_ex_ws: the decode shapes (M <= 16)
// whose k range is split over work-groups keep their fp32 partial sums there;
// large-M shapes with fp16 activations keep the weights decoded to fp16.
extern "C" int64_t dimq_linear_codebook_workspace_bytes(int64_t M, int64_t K, int64_t N, int bits, int x_dtype) {
  const int64_t pd = predecoded_ws_bytes(M, K, N, bits, x_dtype);
  if (pd > 0) return pd;
  if (M <= 0 || M > 16 || K <= 0 || N <= 0 || !(bits == 2 || bits == 3 || bits == 4)) return 0;
  GemmArgs p{};
  p.M = M;
  p.K = K;
  p.N = N;
  p.fast_b = p.vec_a = true;
  if (gemv_direct_ok(p, bits, x_dtype)) return 0;  // no split k
  GemvPlan pl;
  if (!gemv_plan(p, bits, true, pl)) return 0;
  return (gemv_partial_bytes(p, pl) + 255) / 256 * 256;
}

// The arguments of a Linear as the general pre-laid path's plan reads them (no pointers).
static GemmArgs linear_shape_args(int64_t M, int64_t K, int64_t N, int cb_dtype) {
  GemmArgs p{};
  p.M = M;
  p.K = p.ldx = K;
  p.N = p.ldy = N;
  p.cb_dt = cb_dtype;
  p.groups = 1;
  return p;
}

// dimq_linear_codebook_workspace_bytes, or what the general pre-laid path or
// the partial outputs of the large tiles' k ranges need where no other path
// with a workspace takes the shape.
extern "C" int64_t dimq_linear_codebook_full_workspace_bytes(int64_t M, int64_t K, int64_t N, int bits, int x_dtype) {
  const int64_t own = dimq_linear_codebook_workspace_bytes(M, K, N, bits, x_dtype);
  if (own > 0 || M <= 0 || K <= 0 || N <= 0) return own;
  if (!gen_wants_linear(M, K, N, bits)) {
    const int sp = M > 64 && M < 2048 ? big_linear_splits(M, K, N, 7) : 1;
    return sp > 1 ? split_bytes(sp, M, N) : 0;
  }
  const GenPlan g = gen_plan(linear_shape_args(M, K, N, DIMQ_F32), bits, x_dtype, false, true);
  return g.ok ? g.bytes : 0;
}

extern "C" int dimq_linear_codebook_ex_ws(const void* x, int x_dtype, int64_t M, int64_t K, const uint8_t* packed_w,
                                          int64_t packed_numel, int bits, const void* codebook, int cb_dtype,
                                          int64_t cb_rows, int64_t cb_size, const void* bias, int bias_dtype,
                                          int64_t N, void* y, int y_dtype, const void* residual, int residual_dtype,
                                          int activation, int variant, void* workspace, int64_t workspace_bytes,
                                          void* stream) {
  DIMQ_CHECK(workspace_bytes >= 0, "workspace_bytes must be non-negative");
  return linear_codebook_checked(x, x_dtype, M, K, packed_w, packed_numel, bits, codebook, cb_dtype, cb_rows, cb_size,
                                 bias, bias_dtype, N, y, y_dtype, residual, residual_dtype, activation, variant,
                                 stream, workspace, workspace_bytes);
}

extern "C" int64_t dimq_codebook_predecode_bytes(int64_t out_features, int64_t in_features, int bits) {
  return predecoded_w_bytes(out_features, in_features, bits);
}

extern "C" int dimq_codebook_predecode_batch(const DimqPredecodeJob* jobs, int count, void* stream) {
  DIMQ_CHECK(count >= 0 && (count == 0 || jobs != nullptr), "jobs must hold count entries");
  for (int j = 0; j < count; ++j) {
    const DimqPredecodeJob& J = jobs[j];
    if (predecoded_w_bytes(J.out_features, J.in_features, J.bits) == 0)
      return set_error(DIMQ_ERR_UNSUPPORTED, "job %d: pre-decode needs bits 2-4 and in_features %% 32 == 0", j);
    DIMQ_CHECK(J.packed_w != nullptr && J.codebook != nullptr && J.decoded != nullptr, "job %d: null pointer", j);
    DIMQ_CHECK(aligned(J.packed_w, 16), "job %d: packed_w must be 16-byte aligned", j);
    DIMQ_CHECK(aligned(J.decoded, 256), "job %d: decoded must be 256-byte aligned", j);
    DIMQ_CHECK(is_float_dtype(J.cb_dtype), "job %d: codebook must be floating point", j);
    DIMQ_CHECK(J.cb_rows == 1 || J.cb_rows == J.out_features,
               "job %d: codebook must have 1 (per layer) or out_features (per channel) rows", j);
    DIMQ_CHECK(J.cb_size >= 1 && J.cb_size <= (1 << J.bits), "job %d: codebook rows must hold 1 to 2^bits entries", j);
    DIMQ_CHECK(J.packed_numel >= (J.out_features * J.in_features * J.bits + 7) / 8,
               "job %d: packed_weight is too small for out_features * in_features", j);
  }
  return launch_predecode_jobs(jobs, count, as_stream(stream));
}

extern "C" int dimq_linear_codebook_predecoded(const void* x, int x_dtype, int64_t M, int64_t K,
                                               const uint8_t* packed_w, int64_t packed_numel, int bits,
                                               const void* codebook, int cb_dtype, int64_t cb_rows, int64_t cb_size,
                                               const void* bias, int bias_dtype, int64_t N, void* y, int y_dtype,
                                               const void* residual, int residual_dtype, int activation, int variant,
                                               const void* decoded, void* workspace, int64_t workspace_bytes,
                                               void* stream) {
  DIMQ_CHECK(workspace_bytes >= 0, "workspace_bytes must be non-negative");
  DIMQ_CHECK(decoded == nullptr || aligned(decoded, 256), "decoded must be 256-byte aligned");
  return linear_codebook_checked(x, x_dtype, M, K, packed_w, packed_numel, bits, codebook, cb_dtype, cb_rows, cb_size,
                                 bias, bias_dtype, N, y, y_dtype, residual, residual_dtype, activation, variant,
                                 stream, workspace, workspace_bytes, decoded);
}

extern "C" int64_t dimq_linear_codebook_act_workspace_bytes(int64_t M, int64_t K) {
  if (M <= 0 || K <= 0) return 0;
  return (M * K * 4 + 255) / 256 * 256;
}

// Activations replaced by their nearest activation-codebook centre in x's
// dtype (centers[idx].to(x.dtype), quant/dimq.py:217; one element-wise pass
// into the workspace), then the weight-codebook tiles on them, under their
// fp16 range guard: the dequantize-then-MFMA form of the weight x activation
// codebook product.
extern "C" int dimq_linear_codebook_act(const void* x, int x_dtype, int64_t M, int64_t K, const uint8_t* packed_w,
                                        int64_t packed_numel, int bits, const void* codebook, int cb_dtype,
                                        int64_t cb_rows, int64_t cb_size, const float* act_centers, int64_t n_act,
                                        const void* bias, int bias_dtype, int64_t N, void* y, int y_dtype, int variant,
                                        void* workspace, int64_t workspace_bytes, void* stream) {
  DIMQ_CHECK(x_dtype == DIMQ_F32 || x_dtype == DIMQ_F16 || x_dtype == DIMQ_BF16,
             "linear_codebook_act expects fp32, fp16 or bf16 input");
  DIMQ_CHECK(n_act >= 1 && n_act <= 256, "activation codebook must hold between 1 and 256 centres");
  DIMQ_CHECK(act_centers != nullptr, "activation codebook is required");
  DIMQ_CHECK(M >= 0 && N > 0 && K > 0, "linear dimensions must be positive");
  if (M == 0) return DIMQ_OK;
  const int64_t need = dimq_linear_codebook_act_workspace_bytes(M, K);
  DIMQ_CHECK(workspace != nullptr && workspace_bytes >= need && aligned(workspace, 16),
             "workspace must be 16-byte aligned and hold dimq_linear_codebook_act_workspace_bytes bytes");
  // DIMQ_VARIANT_SMALL_M: activation indices into the workspace, then the
  // index x index LUT gather (the weight and activation codebooks' product
  // table formed per work-group); otherwise the dequantize-then-GEMM form,
  // the faster one on MI355X at every M
  const bool gather = variant == DIMQ_VARIANT_SMALL_M && lut_act_supported(M, K, bits, cb_rows, n_act) &&
                      aligned(packed_w, 4) && is_float_dtype(cb_dtype) && (cb_rows == 1 || cb_rows == N) &&
                      cb_size >= 1 && cb_size <= (1 << bits) && packed_numel >= (N * K * bits + 7) / 8;
  if (gather) {
    uint8_t* idx = static_cast<uint8_t*>(workspace);
    int r = dimq_hard_quantize(x, x_dtype, 1, M * K, act_centers, n_act, 0, idx, nullptr, stream);
    if (r != DIMQ_OK) return r;
    DIMQ_CHECK(bias == nullptr || is_float_dtype(bias_dtype), "bias must be floating point");
    DIMQ_CHECK(y_dtype == DIMQ_F32 || y_dtype == DIMQ_F16 || y_dtype == DIMQ_BF16,
               "linear_codebook output dtype must be fp32, fp16 or bf16");
    return launch_lut_act(idx, M, K, packed_w, bits, codebook, cb_dtype, cb_rows, cb_size, act_centers, n_act, x_dtype,
                          bias, bias_dtype, N, y, y_dtype, /*clamp=*/false, as_stream(stream));
  }
  const int rc = launch_act_codebook(x, x_dtype, M * K, act_centers, static_cast<int>(n_act), workspace,
                                     as_stream(stream));
  if (rc != DIMQ_OK) return rc;
  return dimq_linear_codebook_ex(workspace, x_dtype, M, K, packed_w, packed_numel, bits, codebook, cb_dtype, cb_rows, cb_size,
                                 bias, bias_dtype, N, y, y_dtype, nullptr, 0, DIMQ_ACT_NONE, variant, stream);
}

extern "C" int dimq_linear_codebook_ex(const void* x, int x_dtype, int64_t M, int64_t K, const uint8_t* packed_w,
                                       int64_t packed_numel, int bits, const void* codebook, int cb_dtype,
                                       int64_t cb_rows, int64_t cb_size, const void* bias, int bias_dtype, int64_t N,
                                       void* y, int y_dtype, const void* residual, int residual_dtype,
                                       int activation, int variant, void* stream) {
  return linear_codebook_checked(x, x_dtype, M, K, packed_w, packed_numel, bits, codebook, cb_dtype, cb_rows, cb_size,
                                 bias, bias_dtype, N, y, y_dtype, residual, residual_dtype, activation, variant, stream,
                                 nullptr, 0);
}

// Argument checks of the weight-only Linear, then the kernels; `workspace`
// (nullable) may hold the decode GEMV's split-k partial sums.
static int linear_codebook_checked(const void* x, int x_dtype, int64_t M, int64_t K, const uint8_t* packed_w,
                                   int64_t packed_numel, int bits, const void* codebook, int cb_dtype, int64_t cb_rows,
                                   int64_t cb_size, const void* bias, int bias_dtype, int64_t N, void* y, int y_dtype,
                                   const void* residual, int residual_dtype, int activation, int variant, void* stream,
                                   void* workspace, int64_t workspace_bytes, const void* decoded) {
  if (!(bits == 2 || bits == 3 || bits == 4 || bits == 8))
    return set_error(DIMQ_ERR_UNSUPPORTED, "bits must be one of 2, 3, 4, 8 (got %d)", bits);
  DIMQ_CHECK(x_dtype == DIMQ_F32 || x_dtype == DIMQ_F16 || x_dtype == DIMQ_BF16,
             "linear_codebook expects fp32, fp16 or bf16 input");
  DIMQ_CHECK(y_dtype == DIMQ_F32 || y_dtype == DIMQ_F16 || y_dtype == DIMQ_BF16,
             "linear_codebook output dtype must be fp32, fp16 or bf16");
  DIMQ_CHECK(is_float_dtype(cb_dtype), "codebook must be floating point");
  DIMQ_CHECK(bias == nullptr || is_float_dtype(bias_dtype), "bias must be floating point");
  DIMQ_CHECK(M >= 0 && N > 0 && K > 0, "linear dimensions must be positive");
  DIMQ_CHECK(cb_rows == 1 || cb_rows == N, "codebook must have 1 (per layer) or out_features (per channel) rows");
  DIMQ_CHECK(cb_size >= 1 && cb_size <= (1 << bits), "codebook rows must hold between 1 and 2^bits entries");
  DIMQ_CHECK(packed_numel >= (N * K * bits + 7) / 8, "packed_weight is too small for out_features * in_features");
  DIMQ_CHECK(variant >= DIMQ_VARIANT_AUTO && variant <= DIMQ_VARIANT_MFMA, "unknown kernel variant %d", variant);
  DIMQ_CHECK(residual == nullptr || is_float_dtype(residual_dtype), "residual must be floating point");
  DIMQ_CHECK(activation >= DIMQ_ACT_NONE && activation <= DIMQ_ACT_GELU, "unknown activation %d", activation);
  const Epi epi{residual, residual_dtype, activation, residual != nullptr && aligned(residual, 16)};
  return linear_codebook_impl(x, x_dtype, M, K, K, packed_w, bits, codebook, cb_dtype, cb_rows, cb_size, bias,
                              bias_dtype, N, y, y_dtype, N, epi, variant, as_stream(stream), 1.0f, workspace,
                              workspace_bytes, decoded);
}

extern "C" int64_t dimq_linear_lut_workspace_bytes(int64_t M, int64_t in_features, int cb_dtype) {
  if (cb_dtype != DIMQ_F16 || M <= 0 || in_features <= 0) return 0;
  return (M * in_features * 2 + 255) / 256 * 256;
}

// Whether the general pre-laid path takes a W4A4 Linear: in_features off the
// fast tiles' k steps, few rows, and codebooks that are not fp16 -- unless
// their generic A4 tiles (64x128, K % 128 == 0) fill the chip.  Those take per
// k about 28 ns in up to one tile per CU, 36 in up to two, then 66 per 1,024;
// the general path 1.65 ns per 1,000 outputs to lay hi and lo planes out and 8
// per million products of M * N.  4,096 x 4,096: M 1 to 16 107 against 42 us,
// M 512 115 and 94, M 1,024 149 and 168, M 4,096 555 and 640; 8,192 x 8,192:
// M 16 211 and 147, M 512 281 and 362; K 1,024, N 4,096, M 4,096 179 and 164.
static bool lut_wants_gen(int64_t M, int64_t in_features, int64_t out_features, int cb_dtype) {
  if (cb_dtype == DIMQ_F16) return gen_wants_linear(M, in_features, out_features, 4, true);
  if (in_features % kKM != 0 || in_features <= 2048) return true;
  const int64_t tiles = ((M + 63) / 64) * ((out_features + 127) / 128);
  const double a4 = tiles <= device_cus() ? 28.0 : tiles <= 2 * device_cus() ? 36.0 : 0.0645 * tiles;
  return 1.65e-3 * out_features + 8e-6 * M * out_features < a4;
}

// dimq_linear_lut_workspace_bytes, or what the general pre-laid path needs
// where it runs.
extern "C" int64_t dimq_linear_lut_full_workspace_bytes(int x_dtype, int64_t M, int64_t out_features,
                                                        int64_t in_features, int cb_dtype) {
  const int64_t small = dimq_linear_lut_workspace_bytes(M, in_features, cb_dtype);
  if (M <= 0 || out_features <= 0 || in_features <= 0 || !lut_wants_gen(M, in_features, out_features, cb_dtype)) return small;
  const GenPlan g = gen_plan(linear_shape_args(M, in_features, out_features, cb_dtype), 4, x_dtype, true, true);
  return g.ok && g.bytes > small ? g.bytes : small;
}

extern "C" int dimq_linear_lut(const void* x, int x_dtype, int64_t M, const uint8_t* packed_w, int64_t packed_numel,
                               const void* codebook, int cb_dtype, int64_t cb_numel, double act_scale,
                               int64_t act_zp, const void* bias, int bias_dtype, int64_t bias_numel,
                               int64_t out_features, int64_t in_features, float* y, void* stream) {
  return dimq_linear_lut_ws(x, x_dtype, M, packed_w, packed_numel, codebook, cb_dtype, cb_numel, act_scale, act_zp,
                            bias, bias_dtype, bias_numel, out_features, in_features, y, nullptr, 0, stream);
}

// With an fp16 codebook (the reference exporter's default, export.py
// codebook_dtype) and a workspace of M*K fp16: the activations become the
// exact fp16 integers a - zp (one element-wise pass), then the weight-only
// kernels run on them with the 16-entry codebook and act_scale on the
// accumulator, so the call takes the same fast tiles as linear_codebook.
// Otherwise the generic A4 tiles (hi + lo fp16 codebook planes).
// Argument checks of linear_lut, with the messages of the reference's
// TORCH_CHECKs (csrc/dimq_gemm_lut.cu:66-79).
static int check_linear_lut(int x_dtype, int64_t M, int64_t packed_numel, int cb_dtype, int64_t cb_numel,
                            double act_scale, int64_t act_zp, const void* bias, int bias_dtype, int64_t bias_numel,
                            int64_t out_features, int64_t in_features) {
  DIMQ_CHECK(is_float_dtype(x_dtype), "linear_lut expects floating input");
  DIMQ_CHECK(is_float_dtype(cb_dtype), "codebook must be floating point");
  DIMQ_CHECK(cb_numel == 16, "codebook must have 16 entries for W4");
  DIMQ_CHECK(act_scale > 0.0, "act_scale must be positive");
  DIMQ_CHECK(act_zp >= 0 && act_zp <= 15, "act_zero_point must be in [0, 15]");
  DIMQ_CHECK(out_features > 0 && in_features > 0, "linear dimensions must be positive");
  DIMQ_CHECK(M >= 0, "input numel must be divisible by in_features");
  DIMQ_CHECK(packed_numel >= (out_features * in_features + 1) / 2,
             "packed_weight is too small for out_features * in_features");
  if (bias) DIMQ_CHECK(bias_numel == out_features, "bias numel must equal out_features");
  DIMQ_CHECK(bias == nullptr || is_float_dtype(bias_dtype), "bias must be floating point");
  return DIMQ_OK;
}

extern "C" int dimq_linear_lut_ws(const void* x, int x_dtype, int64_t M, const uint8_t* packed_w,
                                  int64_t packed_numel, const void* codebook, int cb_dtype, int64_t cb_numel,
                                  double act_scale, int64_t act_zp, const void* bias, int bias_dtype,
                                  int64_t bias_numel, int64_t out_features, int64_t in_features, float* y,
                                  void* workspace, int64_t workspace_bytes, void* stream) {
  const int rc0 = check_linear_lut(x_dtype, M, packed_numel, cb_dtype, cb_numel, act_scale, act_zp, bias, bias_dtype,
                                   bias_numel, out_features, in_features);
  if (rc0 != DIMQ_OK) return rc0;
  DIMQ_CHECK(workspace_bytes >= 0, "workspace_bytes must be non-negative");
  if (M == 0) return DIMQ_OK;
  if (workspace != nullptr && aligned(workspace, 256) && lut_wants_gen(M, in_features, out_features, cb_dtype)) {
    GemmArgs p = linear_shape_args(M, in_features, out_features, cb_dtype);
    p.x = x;
    p.w = packed_w;
    p.cb = codebook;
    p.cb_rows = 1;
    p.cb_size = 16;
    p.bias = bias;
    p.bias_dt = bias_dtype;
    p.y = y;
    p.y_dt = DIMQ_F32;
    p.acc_scale = p.act_scale = static_cast<float>(act_scale);
    p.act_zp = static_cast<int>(act_zp);
    const GenPlan g = gen_plan(p, 4, x_dtype, true, true);
    if (g.ok && workspace_bytes >= g.bytes) return launch_gen(p, g, 4, x_dtype, workspace, as_stream(stream));
  }
  const int64_t need = dimq_linear_lut_workspace_bytes(M, in_features, cb_dtype);
  if (workspace != nullptr && need > 0 && workspace_bytes >= need && aligned(workspace, 16)) {
    uint16_t* q = static_cast<uint16_t*>(workspace);
    const hipStream_t st = as_stream(stream);
    const int rc = launch_quantize_a4_f16(x, x_dtype, M * in_features, static_cast<float>(act_scale),
                                          static_cast<int>(act_zp), q, st);
    if (rc != DIMQ_OK) return rc;
    return linear_codebook_impl(q, DIMQ_F16, M, in_features, in_features, packed_w, 4, codebook, cb_dtype, 1, 16,
                                bias, bias_dtype, out_features, y, DIMQ_F32, out_features, Epi{}, DIMQ_VARIANT_AUTO,
                                st, static_cast<float>(act_scale));
  }
  GemmArgs p{};
  p.x = x;
  p.M = M;
  p.K = in_features;
  p.ldx = in_features;
  p.w = packed_w;
  p.N = out_features;
  p.cb = codebook;
  p.cb_dt = cb_dtype;
  p.cb_rows = 1;
  p.cb_size = 16;
  p.bias = bias;
  p.bias_dt = bias_dtype;
  p.y = y;
  p.y_dt = DIMQ_F32;
  p.ldy = out_features;
  p.act_scale = static_cast<float>(act_scale);
  p.act_zp = static_cast<int>(act_zp);
  p.fast_b = (in_features % 32 == 0) && aligned(packed_w, 16);
  p.vec_a = aligned(x, 16) && ((in_features * dtype_size(x_dtype)) % 16 == 0);
  p.groups = 1;
  const int tile = (x_dtype != DIMQ_F64) ? gemm_fast_tile(kTile64x32, p, 4) : kTile64x32;
  return dispatch<true>(p, 4, x_dtype, tile, as_stream(stream));
}

extern "C" int dimq_linear_lut_q(const uint16_t* xq, int64_t M, const uint8_t* packed_w, int64_t packed_numel,
                                 const void* codebook, int cb_dtype, int64_t cb_numel, double act_scale,
                                 const void* bias, int bias_dtype, int64_t bias_numel, int64_t out_features,
                                 int64_t in_features, int activation, double out_act_scale, int64_t out_act_zp,
                                 void* y, int y_dtype, void* stream) {
  int rc = check_linear_lut(DIMQ_F16, M, packed_numel, cb_dtype, cb_numel, act_scale, 0, bias, bias_dtype, bias_numel,
                            out_features, in_features);
  if (rc != DIMQ_OK) return rc;
  DIMQ_CHECK(cb_dtype == DIMQ_F16, "linear_lut_q takes the fp16 codebook of the packed export");
  Epi epi;
  rc = lut_q_epilogue(activation, out_act_scale, out_act_zp, y_dtype, epi);
  if (rc != DIMQ_OK) return rc;
  if (M == 0) return DIMQ_OK;
  return linear_codebook_impl(xq, DIMQ_F16, M, in_features, in_features, packed_w, 4, codebook, cb_dtype, 1, 16, bias,
                              bias_dtype, out_features, y, y_dtype, out_features, epi, DIMQ_VARIANT_AUTO,
                              as_stream(stream), static_cast<float>(act_scale));
}

// ---------------------------------------------------------------------------
// dimq_linear_lut_noalloc: dimq_linear_lut_ws with the library's own scratch
// in place of a caller workspace, for callers that cannot allocate.  The
// scratch is one file-scope device array per GPU (a copy on every device the
// library runs on, held until the process ends); host code reaches it only
// through the address hipGetSymbolAddress returns for the current device.
// Every call on a GPU shares that GPU's copy: calls that overlap on one GPU
// (other streams, other host threads) race on it.

constexpr int64_t kNoAllocScratchBytes = 16ll << 20;  // M * in_features <= 8,388,608 fp16 activations

static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

// Device address of `scratch` on the current device, looked up once per
// device with that device current; nullptr (and the HIP error) on failure.
static void* scratch_address(hipError_t* err) {
  static std::mutex mu;
  static void* addr[64] = {};
  int dev = 0;
  *err = hipGetDevice(&dev);
  if (*err != hipSuccess) return nullptr;
  if (dev < 0 || dev >= 64) {
    *err = hipErrorInvalidDevice;
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(mu);
  if (addr[dev] == nullptr) {
    void* p = nullptr;
    *err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (*err != hipSuccess) return nullptr;
    addr[dev] = p;
  }
  return addr[dev];
}

extern "C" int dimq_linear_lut_noalloc(const void* x, int x_dtype, int64_t M, const uint8_t* packed_w,
                                       int64_t packed_numel, const void* codebook, int cb_dtype, int64_t cb_numel,
                                       double act_scale, int64_t act_zp, const void* bias, int bias_dtype,
                                       int64_t bias_numel, int64_t out_features, int64_t in_features, float* y,
                                       void* stream) {
  const int rc = check_linear_lut(x_dtype, M, packed_numel, cb_dtype, cb_numel, act_scale, act_zp, bias, bias_dtype,
                                  bias_numel, out_features, in_features);
  if (rc != DIMQ_OK) return rc;
  const int64_t need = dimq_linear_lut_workspace_bytes(M, in_features, cb_dtype);
  if (need > kNoAllocScratchBytes)
    return set_error(DIMQ_ERR_INVALID,
                     "linear_lut_noalloc: M * in_features = %lld exceeds the scratch limit of %lld activations",
                     (long long)(M * in_features), (long long)(kNoAllocScratchBytes / 2));
  void* ws = nullptr;
  if (need > 0) {
    hipError_t err = hipSuccess;
    ws = scratch_address(&err);
    if (ws == nullptr)
      return set_error(DIMQ_ERR_HIP, "linear_lut_noalloc: hipGetSymbolAddress(scratch): %s", hipGetErrorString(err));
  }
  return dimq_linear_lut_ws(x, x_dtype, M, packed_w, packed_numel, codebook, cb_dtype, cb_numel, act_scale, act_zp,
                            bias, bias_dtype, bias_numel, out_features, in_features, y, ws, need, stream);
}
