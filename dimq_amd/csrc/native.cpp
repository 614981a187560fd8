// dimq_amd._native: the torch side of the hot operators.  Argument checks
// (the reference's TORCH_CHECK messages, csrc/dimq_gemm_lut.cu:66-79,
// csrc/dimq_conv2d_lut.cu:98-134), output and workspace allocation and the
// call into libdimq_hip.so's C ABI on the current stream, registered for the
// CUDA dispatch key in the `dimq` library; and the QAT functions as autograd
// nodes (quant/dimq.py:224-296), whose backward needs no Python.  In Python
// one such call cost 15 to 20 us of host time, more than most of its kernels.
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>
#include <torch/library.h>

#include <optional>
#include <string>
#include <tuple>

#include "../../include/dimq_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

void check_rc(int rc) { TORCH_CHECK(rc == DIMQ_OK, dimq_last_error()); }

std::string dtype_name(at::ScalarType t) { return "torch." + c10::getDtypeNames(t).first; }

int dt(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return DIMQ_F32;
    case at::kHalf: return DIMQ_F16;
    case at::kBFloat16: return DIMQ_BF16;
    case at::kDouble: return DIMQ_F64;
    case at::kByte: return DIMQ_U8;
    default: TORCH_CHECK(false, "unsupported dtype ", dtype_name(t));
  }
}
int dt(const Tensor& t) { return dt(t.scalar_type()); }

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
const uint8_t* u8(const Tensor& t) { return static_cast<const uint8_t*>(t.data_ptr()); }

// The call's device made current, and its current stream there.
struct On {
  c10::OptionalDeviceGuard guard;
  void* stream;
  explicit On(const Tensor& t) : guard(t.device()), stream(c10::hip::getCurrentHIPStream(t.device().index()).stream()) {}
};

// From torch's caching allocator on the current stream (undefined when 0 bytes
// are needed): back-to-back calls reuse one block without a hipMalloc.
Tensor workspace(int64_t bytes, const Tensor& like) {
  return bytes > 0 ? at::empty({bytes}, like.options().dtype(at::kByte)) : Tensor();
}

// The workspace of a layer whose entry point has kernels that need none:
// without room for it the call runs on those (slower) instead of failing.
Tensor spare_workspace(int64_t bytes, const Tensor& like) {
  try {
    return workspace(bytes, like);
  } catch (const c10::OutOfMemoryError&) {
    return Tensor();
  }
}

struct Bias {
  Tensor t;
  void* p = nullptr;
  int dtype = DIMQ_F32;
  int64_t n = 0;
  Bias(const OptTensor& b, int64_t rows, const char* what) {
    if (!b) return;
    TORCH_CHECK(b->is_cuda(), "bias must be CUDA when provided");
    TORCH_CHECK(b->numel() == rows, "bias numel must equal ", what);
    t = b->contiguous();
    p = t.data_ptr();
    dtype = dt(t);
    n = rows;
  }
};

std::pair<int64_t, int64_t> codebook_shape(const Tensor& cb, int64_t n) {
  if (cb.dim() == 2 && cb.size(0) == n && n != 1) return {cb.size(0), cb.size(1)};
  if (cb.dim() == 2 && cb.size(0) == 1) return {1, cb.size(1)};
  if (cb.dim() <= 1) return {1, cb.numel()};
  TORCH_CHECK(false, "codebook must be [K] (per layer) or [out_features, K] (per channel)");
}

std::string tuple_of(at::IntArrayRef s) {
  std::string r = "(";
  for (size_t i = 0; i < s.size(); ++i) r += (i ? ", " : "") + std::to_string(s[i]);
  return r + (s.size() == 1 ? ",)" : ")");
}

// Residual of the fused epilogue, in y's shape, moved into y's memory order.
struct Residual {
  Tensor t;
  void* p = nullptr;
  int dtype = DIMQ_F32;
  Residual(const OptTensor& r, at::IntArrayRef shape, at::MemoryFormat mf) {
    if (!r) return;
    TORCH_CHECK(r->is_cuda(), "residual must be CUDA when provided");
    TORCH_CHECK(r->sizes() == shape, "residual shape ", tuple_of(r->sizes()), " must equal the output shape ",
                tuple_of(shape));
    TORCH_CHECK(r->is_floating_point(), "residual must be floating point");
    t = r->contiguous(mf);
    p = t.data_ptr();
    dtype = dt(t);
  }
};

std::vector<int64_t> out_shape(const Tensor& x, int64_t n) {
  std::vector<int64_t> s = x.sizes().vec();
  s.back() = n;
  return s;
}

int64_t conv_out(int64_t size, int64_t pad, int64_t dil, int64_t k, int64_t stride) {
  if (stride <= 0) return 0;
  const int64_t a = size + 2 * pad - dil * (k - 1) - 1;
  const int64_t q = a >= 0 ? a / stride : -((-a + stride - 1) / stride);  // floor
  return q + 1 > 0 ? q + 1 : 0;
}

// ---- W4A4 ops (csrc/dimq_gemm_lut.cu:58-117, csrc/dimq_conv2d_lut.cu:90-186) ----

Tensor linear_lut(const Tensor& x, const Tensor& packed_w, const Tensor& codebook, double act_scale, int64_t act_zp,
                  const OptTensor& bias, int64_t out_features, int64_t in_features) {
  TORCH_CHECK(x.is_cuda(), "linear_lut expects CUDA input");
  TORCH_CHECK(packed_w.is_cuda(), "linear_lut expects CUDA packed_weight");
  TORCH_CHECK(codebook.is_cuda(), "linear_lut expects CUDA codebook");
  TORCH_CHECK(x.is_floating_point(), "linear_lut expects floating input");
  TORCH_CHECK(packed_w.scalar_type() == at::kByte, "packed_weight must be uint8");
  TORCH_CHECK(codebook.is_floating_point(), "codebook must be floating point");
  TORCH_CHECK(codebook.numel() == 16, "codebook must have 16 entries for W4");
  TORCH_CHECK(out_features > 0 && in_features > 0, "linear dimensions must be positive");
  TORCH_CHECK(x.numel() % in_features == 0, "input numel must be divisible by in_features");
  TORCH_CHECK(x.dim() > 0 && x.size(-1) == in_features, "input last dimension must equal in_features");
  const Tensor xc = x.contiguous(), pw = packed_w.contiguous(), cb = codebook.contiguous();
  const Bias b(bias, out_features, "out_features");
  const int64_t M = xc.numel() / in_features;
  const Tensor y = at::empty(out_shape(x, out_features), x.options().dtype(at::kFloat));
  const On on(xc);
  const Tensor ws = spare_workspace(
      dimq_linear_lut_full_workspace_bytes(dt(xc), M, out_features, in_features, dt(cb)), xc);
  check_rc(dimq_linear_lut_ws(ptr(xc), dt(xc), M, u8(pw), pw.numel(), ptr(cb), dt(cb), cb.numel(), act_scale, act_zp,
                              b.p, b.dtype, b.n, out_features, in_features, static_cast<float*>(y.data_ptr()), ptr(ws),
                              ws.defined() ? ws.numel() : 0, on.stream));
  return y;
}

Tensor conv2d_lut(const Tensor& x, const Tensor& packed_w, const Tensor& codebook, double act_scale, int64_t act_zp,
                  const OptTensor& bias, int64_t out_channels, int64_t in_channels_per_group, int64_t kernel_h,
                  int64_t kernel_w, int64_t stride_h, int64_t stride_w, int64_t pad_h, int64_t pad_w,
                  int64_t dilation_h, int64_t dilation_w, int64_t groups) {
  TORCH_CHECK(x.is_cuda(), "conv2d_lut expects CUDA input");
  TORCH_CHECK(x.dim() == 4, "conv2d_lut expects NCHW input");
  TORCH_CHECK(packed_w.is_cuda(), "conv2d_lut expects CUDA packed_weight");
  TORCH_CHECK(codebook.is_cuda(), "conv2d_lut expects CUDA codebook");
  TORCH_CHECK(x.is_floating_point(), "conv2d_lut expects floating input");
  TORCH_CHECK(packed_w.scalar_type() == at::kByte, "packed_weight must be uint8");
  TORCH_CHECK(codebook.is_floating_point(), "codebook must be floating point");
  const Tensor xc = x.contiguous(), pw = packed_w.contiguous(), cb = codebook.contiguous();
  const int64_t B = xc.size(0), C = xc.size(1), H = xc.size(2), W = xc.size(3);
  const Bias b(bias, out_channels, "out_channels");
  const Tensor y = at::empty({B, out_channels, conv_out(H, pad_h, dilation_h, kernel_h, stride_h),
                              conv_out(W, pad_w, dilation_w, kernel_w, stride_w)}, x.options().dtype(at::kFloat));
  const On on(xc);
  Tensor ws;
  if (y.numel() > 0)
    ws = spare_workspace(dimq_conv2d_lut_full_workspace_bytes(
        dt(xc), B, C, H, W, out_channels, in_channels_per_group, kernel_h, kernel_w, stride_h, stride_w, pad_h, pad_w,
        dilation_h, dilation_w, groups, dt(cb)), xc);
  check_rc(dimq_conv2d_lut_ws(ptr(xc), dt(xc), B, C, H, W, u8(pw), pw.numel(), ptr(cb), dt(cb), cb.numel(), act_scale,
                              act_zp, b.p, b.dtype, b.n, out_channels, in_channels_per_group, kernel_h, kernel_w,
                              stride_h, stride_w, pad_h, pad_w, dilation_h, dilation_w, groups,
                              static_cast<float*>(y.data_ptr()), ptr(ws), ws.defined() ? ws.numel() : 0, on.stream));
  return y;
}

// ---- weight-only ops ----------------------------------------------------------

Tensor linear_codebook(const Tensor& x, const Tensor& packed_w, const Tensor& codebook, int64_t bits,
                       const OptTensor& bias, int64_t out_features, int64_t in_features,
                       std::optional<at::ScalarType> out_dtype, int64_t variant, const OptTensor& residual,
                       int64_t activation, const OptTensor& decoded) {
  TORCH_CHECK(x.is_cuda(), "linear_codebook expects CUDA input");
  TORCH_CHECK(packed_w.is_cuda(), "linear_codebook expects CUDA packed_weight");
  TORCH_CHECK(codebook.is_cuda(), "linear_codebook expects CUDA codebook");
  TORCH_CHECK(x.dim() > 0 && x.size(-1) == in_features, "input last dimension must equal in_features");
  TORCH_CHECK(packed_w.scalar_type() == at::kByte, "packed_weight must be uint8");
  const Tensor xc = x.contiguous(), pw = packed_w.contiguous(), cb = codebook.contiguous();
  const auto [rows, size] = codebook_shape(cb, out_features);
  const Bias b(bias, out_features, "out_features");
  const int64_t M = in_features ? xc.numel() / in_features : 0;
  const std::vector<int64_t> shape = out_shape(x, out_features);
  const Tensor y = at::empty(shape, x.options().dtype(out_dtype.value_or(x.scalar_type())));
  const Residual r(residual, shape, at::MemoryFormat::Contiguous);
  const int nb = static_cast<int>(bits), act = static_cast<int>(activation), var = static_cast<int>(variant);
  const On on(xc);
  const Tensor ws =
      spare_workspace(dimq_linear_codebook_full_workspace_bytes(M, in_features, out_features, nb, dt(xc)), xc);
  const int64_t wsn = ws.defined() ? ws.numel() : 0;
  if (!decoded) {
    check_rc(dimq_linear_codebook_ex_ws(ptr(xc), dt(xc), M, in_features, u8(pw), pw.numel(), nb, ptr(cb), dt(cb), rows,
                                        size, b.p, b.dtype, out_features, ptr(y), dt(y), r.p, r.dtype, act, var,
                                        ptr(ws), wsn, on.stream));
  } else {
    TORCH_CHECK(decoded->is_cuda(), "decoded weights must be CUDA");
    TORCH_CHECK(decoded->scalar_type() == at::kByte &&
                    decoded->numel() >= dimq_codebook_predecode_bytes(out_features, in_features, nb),
                "decoded must be the uint8 buffer predecode_codebook_weights made for this layer");
    check_rc(dimq_linear_codebook_predecoded(ptr(xc), dt(xc), M, in_features, u8(pw), pw.numel(), nb, ptr(cb), dt(cb),
                                             rows, size, b.p, b.dtype, out_features, ptr(y), dt(y), r.p, r.dtype, act,
                                             var, ptr(*decoded), ptr(ws), wsn, on.stream));
  }
  return y;
}

Tensor conv2d_codebook(const Tensor& x, const Tensor& packed_w, const Tensor& codebook, int64_t bits,
                       const OptTensor& bias, int64_t out_channels, int64_t in_channels_per_group, int64_t kernel_h,
                       int64_t kernel_w, int64_t stride_h, int64_t stride_w, int64_t pad_h, int64_t pad_w,
                       int64_t dilation_h, int64_t dilation_w, int64_t groups, std::optional<at::ScalarType> out_dtype,
                       int64_t variant, const OptTensor& prepared_w, const OptTensor& residual, int64_t activation) {
  TORCH_CHECK(x.is_cuda(), "conv2d_codebook expects CUDA input");
  TORCH_CHECK(x.dim() == 4, "conv2d_codebook expects a 4-D input");
  TORCH_CHECK(packed_w.is_cuda(), "conv2d_codebook expects CUDA packed_weight");
  TORCH_CHECK(codebook.is_cuda(), "conv2d_codebook expects CUDA codebook");
  TORCH_CHECK(packed_w.scalar_type() == at::kByte, "packed_weight must be uint8");
  const int64_t B = x.size(0), C = x.size(1), H = x.size(2), W = x.size(3);
  TORCH_CHECK(C == in_channels_per_group * groups, "input channels do not match weight/groups");
  const bool last = !x.is_contiguous() && x.is_contiguous(at::MemoryFormat::ChannelsLast);
  const auto mf = last ? at::MemoryFormat::ChannelsLast : at::MemoryFormat::Contiguous;
  const int layout = last ? DIMQ_NHWC : DIMQ_NCHW;
  const Tensor xc = last ? x : x.contiguous(), pw = packed_w.contiguous(), cb = codebook.contiguous();
  const auto [rows, size] = codebook_shape(cb, out_channels);
  const Bias b(bias, out_channels, "out_channels");
  const Tensor y = at::empty({B, out_channels, conv_out(H, pad_h, dilation_h, kernel_h, stride_h),
                              conv_out(W, pad_w, dilation_w, kernel_w, stride_w)},
                             x.options().dtype(out_dtype.value_or(x.scalar_type())), mf);
  Tensor prep;
  if (prepared_w) {
    TORCH_CHECK(prepared_w->is_cuda(), "prepared_w must be CUDA when provided");
    prep = prepared_w->contiguous();
  }
  const int64_t prep_words = prep.defined() ? prep.numel() : 0;
  const Residual r(residual, y.sizes(), mf);
  const int nb = static_cast<int>(bits), act = static_cast<int>(activation), var = static_cast<int>(variant);
  const On on(xc);
  const Tensor ws = spare_workspace(dimq_conv2d_codebook_workspace_bytes(
      dt(xc), layout, B, C, H, W, nb, prep_words > 0, dt(cb), rows, size, out_channels, kernel_h, kernel_w, stride_h,
      stride_w, pad_h, pad_w, dilation_h, dilation_w, groups, dt(y), layout, r.p != nullptr, act, var), xc);
  check_rc(dimq_conv2d_codebook_ex_ws(ptr(xc), dt(xc), layout, B, C, H, W, u8(pw), pw.numel(), nb,
                                      static_cast<const uint32_t*>(ptr(prep)), prep_words, ptr(cb), dt(cb), rows, size,
                                      b.p, b.dtype, out_channels, kernel_h, kernel_w, stride_h, stride_w, pad_h, pad_w,
                                      dilation_h, dilation_w, groups, ptr(y), dt(y), layout, r.p, r.dtype, act, var,
                                      ptr(ws), ws.defined() ? ws.numel() : 0, on.stream));
  return y;
}

// ---- codec, nearest centres, support ops ----------------------------------------

Tensor pack_bits(const Tensor& indices, int64_t bits) {
  TORCH_CHECK(indices.is_cuda(), "pack_bits expects a CUDA tensor");
  TORCH_CHECK(indices.scalar_type() == at::kByte, "pack_bits expects uint8 indices");
  const Tensor flat = indices.contiguous();
  const int64_t bytes = flat.numel() * bits + 7;
  const Tensor out = at::empty({bytes >= 0 ? bytes / 8 : 0}, flat.options());
  const On on(flat);
  check_rc(dimq_pack_bits(u8(flat), flat.numel(), static_cast<int>(bits), static_cast<uint8_t*>(out.data_ptr()),
                          on.stream));
  return out;
}

Tensor unpack_bits(const Tensor& packed, int64_t numel, int64_t bits) {
  TORCH_CHECK(packed.is_cuda(), "unpack_bits expects a CUDA tensor");
  TORCH_CHECK(packed.scalar_type() == at::kByte, "unpack_bits expects uint8 packed data");
  TORCH_CHECK(numel >= 0, "numel must be non-negative");
  const Tensor flat = packed.contiguous();
  const Tensor out = at::empty({numel}, flat.options());
  const On on(flat);
  check_rc(dimq_unpack_bits(u8(flat), flat.numel(), numel, static_cast<int>(bits),
                            static_cast<uint8_t*>(out.data_ptr()), on.stream));
  return out;
}

std::tuple<Tensor, Tensor> hard_quantize(const Tensor& w, const Tensor& centers, bool per_channel) {
  TORCH_CHECK(w.is_cuda(), "hard_quantize expects a CUDA tensor");
  TORCH_CHECK(centers.is_cuda(), "hard_quantize expects CUDA centers");
  Tensor wc = w.contiguous();
  const auto st = wc.scalar_type();
  if (st != at::kFloat && st != at::kHalf && st != at::kBFloat16) wc = wc.to(at::kFloat);
  const Tensor c = centers.detach().to(at::kFloat).contiguous();
  if (per_channel)
    TORCH_CHECK(c.dim() == 2 && wc.dim() > 0 && c.size(0) == wc.size(0),
                "per-channel centers must be [out_channels, K]");
  const int64_t rows = per_channel ? c.size(0) : 1, K = per_channel ? c.size(1) : c.numel();
  const Tensor idx = at::empty(wc.sizes(), wc.options().dtype(at::kByte));
  const Tensor vals = at::empty(wc.sizes(), wc.options());
  const On on(wc);
  check_rc(dimq_hard_quantize(ptr(wc), dt(wc), rows, rows ? wc.numel() / rows : 0,
                              static_cast<const float*>(ptr(c)), K, per_channel, static_cast<uint8_t*>(ptr(idx)),
                              ptr(vals), on.stream));
  return {idx, vals};
}

Tensor layer_norm(const Tensor& x, int64_t D, const OptTensor& weight, const OptTensor& bias, double eps,
                  std::optional<at::ScalarType> out_dtype) {
  TORCH_CHECK(x.is_cuda(), "layer_norm expects CUDA input");
  const auto half = [](at::ScalarType t) { return t == at::kHalf || t == at::kBFloat16; };
  TORCH_CHECK(half(x.scalar_type()), "layer_norm expects fp16 or bf16 input");
  TORCH_CHECK(x.dim() > 0 && x.size(-1) == D, "layer_norm: last input dimension must equal the normalized size");
  Tensor xv = x.dim() != 2 ? x.reshape({-1, D}) : x;
  if (xv.stride(-1) != 1 || xv.stride(0) % 8 != 0 || reinterpret_cast<uintptr_t>(xv.data_ptr()) % 16 != 0)
    xv = xv.contiguous();
  Tensor w, b;
  for (const OptTensor* t : {&weight, &bias}) {
    if (!*t) continue;
    TORCH_CHECK((*t)->is_cuda(), "layer_norm weight and bias must be CUDA tensors");
    TORCH_CHECK((*t)->numel() == D, "layer_norm weight and bias must have the normalized size");
  }
  if (weight) w = weight->contiguous();
  if (bias) b = (weight ? bias->to(weight->scalar_type()) : *bias).contiguous();
  const int wdt = w.defined() ? dt(w) : b.defined() ? dt(b) : static_cast<int>(DIMQ_F32);
  const at::ScalarType odt = out_dtype.value_or(x.scalar_type());
  TORCH_CHECK(half(odt), "layer_norm writes fp16 or bf16 output");
  const Tensor y = at::empty(x.sizes(), x.options().dtype(odt));
  const On on(x);
  check_rc(dimq_layer_norm_ex(ptr(xv), dt(xv), xv.size(0), D, xv.stride(0), ptr(w), ptr(b), wdt, eps, ptr(y), dt(y),
                              on.stream));
  return y;
}

Tensor max_pool2d_nhwc(const Tensor& x, int64_t kernel_h, int64_t kernel_w, int64_t stride_h, int64_t stride_w,
                       int64_t pad_h, int64_t pad_w) {
  TORCH_CHECK(x.is_cuda(), "max_pool2d expects CUDA input");
  TORCH_CHECK(x.dim() == 4 && x.is_contiguous(at::MemoryFormat::ChannelsLast),
              "max_pool2d expects a channels-last 4-D input");
  TORCH_CHECK(x.scalar_type() == at::kHalf || x.scalar_type() == at::kBFloat16,
              "max_pool2d expects fp16 or bf16 input");
  const Tensor y = at::empty({x.size(0), x.size(1), conv_out(x.size(2), pad_h, 1, kernel_h, stride_h),
                              conv_out(x.size(3), pad_w, 1, kernel_w, stride_w)},
                             x.options(), at::MemoryFormat::ChannelsLast);
  const On on(x);
  check_rc(dimq_max_pool2d_nhwc(ptr(x), dt(x), x.size(0), x.size(1), x.size(2), x.size(3), kernel_h, kernel_w,
                                stride_h, stride_w, pad_h, pad_w, ptr(y), on.stream));
  return y;
}

// ---- QAT functions ---------------------------------------------------------------

struct QatInputs {
  Tensor w, c;
  QatInputs(const Tensor& weights, const Tensor& centers) {
    TORCH_CHECK(weights.is_cuda(), "QAT kernels expect CUDA weights");
    TORCH_CHECK(centers.is_cuda(), "QAT kernels expect CUDA centers");
    const auto st = weights.scalar_type();
    TORCH_CHECK(st == at::kFloat || st == at::kHalf || st == at::kBFloat16 || st == at::kDouble,
                "weights must be fp32, fp16, bf16 or fp64");
    w = weights.detach().contiguous();
    c = centers.detach().reshape({-1}).to(at::kFloat).contiguous();
    TORCH_CHECK_VALUE(c.numel() != 0, "centers must be non-empty");
    TORCH_CHECK(c.numel() <= 256, "at most 256 centers are supported");
  }
  int64_t n() const { return w.numel(); }
  int64_t K() const { return c.numel(); }
  const float* cp() const { return static_cast<const float*>(c.data_ptr()); }
  Tensor ws() const { return workspace(dimq_qat_workspace_bytes(n(), K()), w); }
  Tensor fp32(at::IntArrayRef shape) const { return at::empty(shape, w.options().dtype(at::kFloat)); }
};

float* f32(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// w + (w_hard - w).detach(): the hard values forward, the identity to w
// backward, nothing to the centres.
struct HardSte : torch::autograd::Function<HardSte> {
  static Tensor forward(AutogradContext*, const Tensor& w, const Tensor& centers) {
    const Tensor v = std::get<1>(hard_quantize(w.detach(), centers.detach().reshape({-1}), false));
    return v.reshape(w.sizes()).to(w.scalar_type());
  }
  static variable_list backward(AutogradContext*, variable_list g) { return {g[0], Tensor()}; }
};

struct SoftDequantize : torch::autograd::Function<SoftDequantize> {
  static Tensor forward(AutogradContext* ctx, const Tensor& w, const Tensor& centers, double tau) {
    const QatInputs in(w, centers);
    const Tensor out = at::empty_like(in.w), aux = in.fp32({in.n(), 2});
    const On on(in.w);
    check_rc(dimq_soft_dequantize_forward(ptr(in.w), dt(in.w), in.n(), in.cp(), in.K(), tau, ptr(out), f32(aux),
                                          on.stream));
    ctx->save_for_backward({w, centers, aux});
    ctx->saved_data["tau"] = tau;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const QatInputs in(saved[0], saved[1]);
    const Tensor go = grads[0].detach().contiguous();
    const Tensor gw = at::empty_like(in.w), gc = in.fp32({in.K()}), ws = in.ws();
    const On on(in.w);
    check_rc(dimq_soft_dequantize_backward(ptr(in.w), dt(in.w), in.n(), in.cp(), in.K(),
                                           ctx->saved_data["tau"].toDouble(), f32(saved[2]), ptr(go), dt(go), ptr(gw),
                                           dt(gw), f32(gc), ptr(ws), ws.numel(), on.stream));
    return {gw, gc.to(saved[1].scalar_type()).reshape(saved[1].sizes()), Tensor()};
  }
};

struct SoftminLoss : torch::autograd::Function<SoftminLoss> {
  static Tensor forward(AutogradContext* ctx, const Tensor& w, const Tensor& centers, double tau, bool mean) {
    const QatInputs in(w, centers);
    const Tensor aux = in.fp32({in.n(), 2}), loss = in.fp32({}), ws = in.ws();
    const On on(in.w);
    check_rc(dimq_softmin_loss_forward(ptr(in.w), dt(in.w), in.n(), in.cp(), in.K(), tau, mean, f32(aux), f32(loss),
                                       ptr(ws), ws.numel(), on.stream));
    ctx->save_for_backward({w, centers, aux});
    ctx->saved_data["tau"] = tau;
    ctx->saved_data["mean"] = mean;
    return loss;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const QatInputs in(saved[0], saved[1]);
    Tensor g = grads[0].detach();
    if (ctx->saved_data["mean"].toBool()) g = g / static_cast<double>(in.n() > 1 ? in.n() : 1);
    g = g.reshape({}).to(at::kFloat).contiguous();
    const Tensor gw = at::empty_like(in.w), gc = in.fp32({in.K()}), ws = in.ws();
    const On on(in.w);
    check_rc(dimq_softmin_loss_backward(ptr(in.w), dt(in.w), in.n(), in.cp(), in.K(), ctx->saved_data["tau"].toDouble(),
                                        0, f32(saved[2]), f32(g), ptr(gw), dt(gw), f32(gc), ptr(ws), ws.numel(),
                                        on.stream));
    return {gw, gc.to(saved[1].scalar_type()).reshape(saved[1].sizes()), Tensor(), Tensor()};
  }
};

struct SeparationLoss : torch::autograd::Function<SeparationLoss> {
  static Tensor forward(AutogradContext* ctx, const Tensor& w, const Tensor& centers, double eta, double eps) {
    const QatInputs in(w, centers);
    const Tensor loss = in.fp32({}), gc = in.fp32({in.K()}), ws = in.ws();
    const On on(in.w);
    check_rc(dimq_separation_loss(ptr(in.w), dt(in.w), in.n(), in.cp(), in.K(), eta, eps, f32(loss), f32(gc), ptr(ws),
                                  ws.numel(), on.stream));
    ctx->save_for_backward({gc});
    ctx->saved_data["shape"] = centers.sizes().vec();
    ctx->saved_data["dtype"] = static_cast<int64_t>(centers.scalar_type());
    return loss;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto shape = ctx->saved_data["shape"].toIntVector();
    const auto type = static_cast<at::ScalarType>(ctx->saved_data["dtype"].toInt());
    return {Tensor(), (grads[0] * ctx->get_saved_variables()[0]).to(type).reshape(shape), Tensor(), Tensor()};
  }
};

}  // namespace

TORCH_LIBRARY_FRAGMENT(dimq, m) {
  // the first two verbatim from dimq_cuda_backend/csrc/dimq_ops.cpp:38-43
  m.def("linear_lut(Tensor x, Tensor packed_w, Tensor codebook, float act_scale, int act_zp, Tensor? bias, "
        "int out_features, int in_features) -> Tensor");
  m.def("conv2d_lut(Tensor x, Tensor packed_w, Tensor codebook, float act_scale, int act_zp, Tensor? bias, "
        "int out_channels, int in_channels_per_group, int kernel_h, int kernel_w, int stride_h, int stride_w, "
        "int pad_h, int pad_w, int dilation_h, int dilation_w, int groups) -> Tensor");
  m.def("pack_bits(Tensor indices, int bits) -> Tensor");
  m.def("unpack_bits(Tensor packed, int numel, int bits) -> Tensor");
  m.def("hard_quantize(Tensor w, Tensor centers, bool per_channel) -> (Tensor, Tensor)");
  m.def("linear_codebook(Tensor x, Tensor packed_w, Tensor codebook, int bits, Tensor? bias, int out_features, "
        "int in_features, ScalarType? out_dtype=None, int variant=0, Tensor? residual=None, int activation=0, "
        "Tensor? decoded=None) -> Tensor");
  m.def("conv2d_codebook(Tensor x, Tensor packed_w, Tensor codebook, int bits, Tensor? bias, int out_channels, "
        "int in_channels_per_group, int kernel_h, int kernel_w, int stride_h, int stride_w, int pad_h, int pad_w, "
        "int dilation_h, int dilation_w, int groups, ScalarType? out_dtype=None, int variant=0, "
        "Tensor? prepared_w=None, Tensor? residual=None, int activation=0) -> Tensor");
  m.def("layer_norm(Tensor x, int normalized_size, Tensor? weight, Tensor? bias, float eps, "
        "ScalarType? out_dtype=None) -> Tensor");
  m.def("max_pool2d_nhwc(Tensor x, int kernel_h, int kernel_w, int stride_h, int stride_w, int pad_h, int pad_w) "
        "-> Tensor");
}

TORCH_LIBRARY_IMPL(dimq, CUDA, m) {
  m.impl("linear_lut", linear_lut);
  m.impl("conv2d_lut", conv2d_lut);
  m.impl("pack_bits", pack_bits);
  m.impl("unpack_bits", unpack_bits);
  m.impl("hard_quantize", hard_quantize);
  m.impl("linear_codebook", linear_codebook);
  m.impl("conv2d_codebook", conv2d_codebook);
  m.impl("layer_norm", layer_norm);
  m.impl("max_pool2d_nhwc", max_pool2d_nhwc);
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  namespace py = pybind11;
  using Unlocked = py::call_guard<py::gil_scoped_release>;
  m.def("linear_lut", &linear_lut, Unlocked());
  m.def("conv2d_lut", &conv2d_lut, Unlocked());
  m.def("hard_ste", [](const Tensor& w, const Tensor& c) { return HardSte::apply(w, c); }, Unlocked());
  m.def("soft_dequantize",
        [](const Tensor& w, const Tensor& c, double tau) { return SoftDequantize::apply(w, c, tau); }, Unlocked());
  m.def("softmin_loss",
        [](const Tensor& w, const Tensor& c, double tau, bool mean) { return SoftminLoss::apply(w, c, tau, mean); },
        Unlocked());
  m.def("separation_loss",
        [](const Tensor& w, const Tensor& c, double eta, double eps) { return SeparationLoss::apply(w, c, eta, eps); },
        Unlocked());
}
