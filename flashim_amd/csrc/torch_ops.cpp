// The C entry points as torch operators of the namespace flashim_amd: each allocates its outputs with torch's caching
// allocator, makes one C call on the current stream of its input's device and raises on a nonzero status. Registered in
// C++, an eager call takes torch's C++ dispatcher only (a Python custom op costs about 10 us a call on the host, more
// than a small layer's kernel); the fakes stay in library.py. Arguments arrive normalized by the Python impls (dtypes,
// contiguity, devices); 1-byte float formats cross as they are or as their uint8 views (the bodies read bytes), and come
// back as uint8.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/pybind11.h>
#include <torch/csrc/autograd/VariableTypeUtils.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/library.h>

#include <array>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/flashim_amd.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

constexpr int64_t BLOCK = 32;

hipStream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

template <typename T>
T* ptr(const Tensor& t) { return static_cast<T*>(t.data_ptr()); }
template <typename T>
T* ptr(const OptTensor& t) { return t ? static_cast<T*>(t->data_ptr()) : nullptr; }

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return 0;
    case at::kBFloat16: return 1;
    case at::kHalf: return 2;
    default: TORCH_CHECK_TYPE(false, "unsupported dtype ", t.scalar_type());
  }
}

int bias_code(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? 1 : 0; }
int bias_code(const OptTensor& t) { return t && t->scalar_type() == at::kBFloat16 ? 1 : 0; }

// Status 99 as the package's own exception, raised here so that compiled graphs, which call the operators themselves, see
// its type too.
[[noreturn]] void raise_unsupported(const std::string& message) {
  pybind11::gil_scoped_acquire gil;
  PyErr_SetString(pybind11::module_::import("flashim_amd._lib").attr("UnsupportedShape").ptr(), message.c_str());
  throw pybind11::error_already_set();
}

template <typename... What>
void check(int code, const What&... what) {
  if (code == FIM_OK) return;
  if (code == FIM_ERR_UNSUPPORTED) raise_unsupported(c10::str(what..., ": no HIP kernel for this shape/layout (code 99)"));
  TORCH_CHECK(false, what..., " launch failed (code ", code, ")");
}

// size() and stride() of the leading dimensions would read an input of more dimensions as one of fewer
void check_dims(const Tensor& t, int64_t dims, const char* what) {
  TORCH_CHECK_VALUE(t.dim() == dims, what, ": expected ", dims, " dimensions, got shape ", t.sizes());
}

Tensor empty(at::IntArrayRef sizes, const Tensor& like, at::ScalarType dtype) {
  return at::empty(sizes, like.options().dtype(dtype).requires_grad(false).memory_format(std::nullopt));
}

// [..., C] as [B, H, W, C] sizes and strides, copying only where leading dimensions do not merge.
struct View4 {
  Tensor t;
  std::array<int64_t, 4> n{1, 1, 1, 1}, s{0, 0, 0, 0};
  explicit View4(const Tensor& x) : t(x) {
    if (t.dim() > 4) t = t.reshape({-1, t.size(-3), t.size(-2), t.size(-1)});
    const int64_t d = t.dim(), pad = 4 - d;
    for (int64_t i = 0; i < d; ++i) {
      n[pad + i] = t.size(i);
      s[pad + i] = t.stride(i);
    }
    for (int64_t i = pad - 1; i >= 0; --i) s[i] = i == 3 ? 1 : n[i + 1] * s[i + 1];  // as unsqueeze does
  }
};

#define FIM_VIEW4(v) v.n[0], v.n[1], v.n[2], v.n[3], v.s[0], v.s[1], v.s[2], v.s[3]

std::vector<int64_t> padded_sizes(const Tensor& value, int64_t padded) {
  auto sizes = value.sizes().vec();
  if (!sizes.empty()) sizes.pop_back();
  sizes.push_back(padded);
  return sizes;
}

Tensor quantize_mxfp8(const Tensor& value, const Tensor& exponent, int64_t padded) {
  const c10::DeviceGuard guard(value.device());
  Tensor out = empty(padded_sizes(value, padded), value, at::kByte);
  const View4 v(value);
  check(fim_quantize_mxfp8(v.t.data_ptr(), dtype_code(value), FIM_VIEW4(v), ptr<const int8_t>(exponent),
                           ptr<uint8_t>(out), padded, stream_of(value)),
        "quantize_mxfp8 ", value.sizes());
  return out;
}

Tensor gelu_quantize_mxfp8(const Tensor& value, const Tensor& exponent, int64_t padded, const OptTensor& input_bias,
                           bool tanh) {
  const c10::DeviceGuard guard(value.device());
  Tensor out = empty(padded_sizes(value, padded), value, at::kByte);
  const View4 v(value);
  check(fim_gelu_quantize_mxfp8(v.t.data_ptr(), dtype_code(value), FIM_VIEW4(v), tanh, ptr<const float>(input_bias),
                                ptr<const int8_t>(exponent), ptr<uint8_t>(out), padded, stream_of(value)),
        "gelu_quantize_mxfp8 ", value.sizes());
  return out;
}

Tensor quantize_int8(const Tensor& value, const Tensor& scale, const OptTensor& channel_scale) {
  const c10::DeviceGuard guard(value.device());
  Tensor out = empty(value.sizes(), value, at::kChar);
  const View4 v(value);
  check(fim_quantize_int8(v.t.data_ptr(), dtype_code(value), FIM_VIEW4(v), ptr<const float>(scale),
                          ptr<const float>(channel_scale), ptr<int8_t>(out), stream_of(value)),
        "quantize_int8 ", value.sizes());
  return out;
}

Tensor gelu_quantize_int8(const Tensor& value, const Tensor& scale, bool tanh) {
  const c10::DeviceGuard guard(value.device());
  Tensor out = empty(value.sizes(), value, at::kChar);
  const View4 v(value);
  check(fim_gelu_quantize_int8(v.t.data_ptr(), dtype_code(value), FIM_VIEW4(v), tanh, ptr<const float>(scale),
                               ptr<int8_t>(out), stream_of(value)),
        "gelu_quantize_int8 ", value.sizes());
  return out;
}

// Swizzled scales: whole 128-row x 4-block tiles; the bytes past the matrix are zero.
Tensor swizzled_scales(int64_t rows, int64_t groups, const Tensor& like) {
  Tensor t = empty({(rows + 127) / 128 * 128 * ((groups + 3) / 4 * 4)}, like, at::kByte);
  if (rows % 128 || groups % 4) t.zero_();
  return t;
}

std::tuple<Tensor, Tensor> quantize_mxfp8_dynamic(const Tensor& value_in, bool swizzled) {
  check_dims(value_in, 2, "quantize_mxfp8_dynamic");
  const c10::DeviceGuard guard(value_in.device());
  Tensor value = value_in;
  if (reinterpret_cast<uintptr_t>(value.data_ptr()) % 16)  // the kernel reads 16-byte rows
    value = value.clone(at::MemoryFormat::Contiguous);
  const int64_t rows = value.size(0), cols = value.size(1), groups = cols / BLOCK;
  Tensor out = empty({rows, cols}, value, at::kByte);
  Tensor scales = swizzled ? swizzled_scales(rows, groups, value) : empty({rows, groups}, value, at::kChar);
  check(fim_quantize_mxfp8_dynamic(value.data_ptr(), dtype_code(value), rows, cols, value.stride(0), ptr<uint8_t>(out),
                                   swizzled ? nullptr : ptr<int8_t>(scales), swizzled ? ptr<uint8_t>(scales) : nullptr,
                                   stream_of(value)),
        "quantize_mxfp8_dynamic ", rows, "x", cols);
  return {out, scales};
}

std::tuple<Tensor, Tensor> quantize_int8_rows(const Tensor& value, bool reciprocal) {
  check_dims(value, 2, "quantize_int8_rows");
  const c10::DeviceGuard guard(value.device());
  const int64_t rows = value.size(0), k = value.size(1);
  Tensor q = empty({rows, k}, value, at::kChar), scale = empty({rows}, value, at::kFloat);
  check(fim_quantize_int8_rows(value.data_ptr(), dtype_code(value), rows, k, value.stride(0), reciprocal, ptr<int8_t>(q),
                               ptr<float>(scale), stream_of(value)),
        "quantize_int8_rows ", rows, "x", k);
  return {q, scale};
}

Tensor calibrate_block32(const Tensor& matrix) {
  check_dims(matrix, 2, "calibrate_block32");
  const c10::DeviceGuard guard(matrix.device());
  const int64_t rows = matrix.size(0), channels = matrix.size(1), groups = (channels + BLOCK - 1) / BLOCK;
  Tensor workspace = empty({groups}, matrix, at::kInt), exponent = empty({groups}, matrix, at::kChar);
  check(fim_calibrate_block32(matrix.data_ptr(), dtype_code(matrix), rows, channels, matrix.stride(0),
                              ptr<uint32_t>(workspace), ptr<int8_t>(exponent), stream_of(matrix)),
        "calibrate_block32");
  return exponent;
}

struct Residual {
  const void* data = nullptr;
  int code = 0;
  int64_t channels = 0;
  std::array<int64_t, 4> strides{};
  const int64_t* stride_ptr = nullptr;
  explicit Residual(const OptTensor& r) {
    if (!r) return;
    data = r->data_ptr();
    code = dtype_code(*r);
    channels = r->size(-1);
    for (int64_t i = 0; i < r->dim() && i < 4; ++i) strides[i] = r->stride(i);
    stride_ptr = strides.data();
  }
};

// kh .. dw of a convolution call as the C ABI takes them, and its output size
struct Geometry {
  int kh, kw, sh, sw, ph, pw, dh, dw;
  int64_t out(int64_t n, int k, int s, int p, int d) const {  // Python's floor division
    const int64_t a = n + 2 * p - static_cast<int64_t>(d) * (k - 1) - 1;
    return (a >= 0 ? a / s : -((-a + s - 1) / s)) + 1;
  }
  int64_t ho(int64_t h) const { return out(h, kh, sh, ph, dh); }
  int64_t wo(int64_t w) const { return out(w, kw, sw, pw, dw); }
};

#define FIM_GEO_PARAMS int64_t kh, int64_t kw, int64_t sh, int64_t sw, int64_t ph, int64_t pw, int64_t dh, int64_t dw
#define FIM_GEO Geometry { (int)kh, (int)kw, (int)sh, (int)sw, (int)ph, (int)pw, (int)dh, (int)dw }
#define FIM_GEO_ARGS(g) g.kh, g.kw, g.sh, g.sw, g.ph, g.pw, g.dh, g.dw

Tensor int8_conv2d(const Tensor& x, const Tensor& weight, const Tensor& a_scale, const Tensor& w_scale,
                   const OptTensor& bias, FIM_GEO_PARAMS, bool relu, bool gelu, const OptTensor& residual,
                   const OptTensor& out_scale) {
  check_dims(x, 4, "int8_conv2d");
  TORCH_CHECK_INDEX(!residual || residual->dim() <= 4, "int8_conv2d: residual of shape ", residual->sizes());
  const c10::DeviceGuard guard(x.device());
  const Geometry g = FIM_GEO;
  const int64_t b = x.size(0), h = x.size(1), w = x.size(2), cin = x.size(3), cout = weight.size(0);
  TORCH_CHECK(sh > 0 && sw > 0, "int8_conv2d: strides must be positive");
  Tensor out = empty({b, g.ho(h), g.wo(w), cout}, x, out_scale ? at::kChar : at::kBFloat16);
  const Residual r(residual);
  check(fim_int8_conv2d(ptr<const int8_t>(x), b, h, w, cin, ptr<const int8_t>(weight), cout, ptr<const float>(a_scale),
                        ptr<const float>(w_scale), ptr<const void>(bias), bias_code(bias), FIM_GEO_ARGS(g), relu, gelu,
                        r.data, r.code, r.channels, r.stride_ptr, ptr<const float>(out_scale), out.data_ptr(),
                        stream_of(x)),
        "int8_conv2d ", x.sizes(), " -> ", cout, " k", kh, "x", kw);
  return out;
}

std::tuple<Tensor, Tensor> int8_conv2d_maxpool(const Tensor& x, const Tensor& weight, const Tensor& a_scale,
                                               const Tensor& w_scale, const OptTensor& bias, FIM_GEO_PARAMS, bool relu,
                                               const Tensor& out_scale) {
  check_dims(x, 4, "int8_conv2d_maxpool");
  const c10::DeviceGuard guard(x.device());
  const Geometry g = FIM_GEO;
  const int64_t b = x.size(0), h = x.size(1), w = x.size(2), cin = x.size(3), cout = weight.size(0);
  TORCH_CHECK(sh > 0 && sw > 0, "int8_conv2d_maxpool: strides must be positive");
  const int64_t ho = g.ho(h), wo = g.wo(w);
  Tensor out = empty({b, ho, wo, cout}, x, at::kBFloat16), pooled = empty({b, ho / 2, wo / 2, cout}, x, at::kChar);
  check(fim_int8_conv2d_maxpool(ptr<const int8_t>(x), b, h, w, cin, ptr<const int8_t>(weight), cout,
                                ptr<const float>(a_scale), ptr<const float>(w_scale), ptr<const void>(bias),
                                bias_code(bias), FIM_GEO_ARGS(g), relu, ptr<const float>(out_scale), out.data_ptr(),
                                ptr<int8_t>(pooled), stream_of(x)),
        "int8_conv2d_maxpool ", x.sizes(), " -> ", cout, " k", kh, "x", kw);
  return {out, pooled};
}

Tensor mxfp8_conv2d(const Tensor& x, const Tensor& channel_exponent, const Tensor& weight, const Tensor& weight_exponent,
                    const OptTensor& bias, FIM_GEO_PARAMS, bool relu, bool gelu, const OptTensor& residual,
                    const OptTensor& out_exponent) {
  check_dims(x, 4, "mxfp8_conv2d");
  TORCH_CHECK_INDEX(!residual || residual->dim() <= 4, "mxfp8_conv2d: residual of shape ", residual->sizes());
  const c10::DeviceGuard guard(x.device());
  const Geometry g = FIM_GEO;
  const int64_t b = x.size(0), h = x.size(1), w = x.size(2), cin = x.size(3), cout = weight.size(0);
  TORCH_CHECK(sh > 0 && sw > 0, "mxfp8_conv2d: strides must be positive");
  Tensor out = empty({b, g.ho(h), g.wo(w), cout}, x, out_exponent ? at::kByte : at::kBFloat16);
  const Residual r(residual);
  check(fim_mxfp8_conv2d(ptr<const uint8_t>(x), b, h, w, cin, ptr<const int8_t>(channel_exponent),
                         ptr<const uint8_t>(weight), cout, ptr<const int8_t>(weight_exponent), ptr<const void>(bias),
                         bias_code(bias), FIM_GEO_ARGS(g), relu, gelu, r.data, r.code, r.channels, r.stride_ptr,
                         ptr<const int8_t>(out_exponent), out.data_ptr(), stream_of(x)),
        "mxfp8_conv2d ", x.sizes(), " -> ", cout, " k", kh, "x", kw);
  return out;
}

Tensor int8_linear(const Tensor& a, const Tensor& weight, const Tensor& a_scale, const Tensor& w_scale,
                   const OptTensor& bias, bool relu, bool gelu, const OptTensor& residual) {
  check_dims(a, 2, "int8_linear");
  const c10::DeviceGuard guard(a.device());
  const int64_t m = a.size(0), k = a.size(1), n = weight.size(0);
  const bool per_row = a_scale.numel() != 1;
  Tensor out = empty({m, n}, a, at::kBFloat16);
  const Residual r(residual);
  check(fim_int8_linear(ptr<const int8_t>(a), m, k, ptr<const int8_t>(weight), n,
                        per_row ? nullptr : ptr<const float>(a_scale), per_row ? ptr<const float>(a_scale) : nullptr,
                        ptr<const float>(w_scale), ptr<const void>(bias), bias_code(bias), relu, gelu, r.data, r.code,
                        r.channels, r.strides[0], nullptr, out.data_ptr(), stream_of(a)),
        "int8_linear ", m, "x", k, " -> ", n);
  return out;
}

void int8_linear_quantize_(const Tensor& a, const Tensor& weight, const Tensor& a_scale, const Tensor& w_scale,
                           const OptTensor& bias, const Tensor& out_scale, const Tensor& out) {
  check_dims(a, 2, "int8_linear_quantize_");
  const c10::DeviceGuard guard(a.device());
  const int64_t m = a.size(0), k = a.size(1), n = weight.size(0);
  const bool per_row = a_scale.numel() != 1;
  check(fim_int8_linear_quantize(ptr<const int8_t>(a), m, k, ptr<const int8_t>(weight), n,
                                 per_row ? nullptr : ptr<const float>(a_scale),
                                 per_row ? ptr<const float>(a_scale) : nullptr, ptr<const float>(w_scale),
                                 ptr<const void>(bias), bias_code(bias), ptr<const float>(out_scale), ptr<int8_t>(out),
                                 out.stride(0), stream_of(a)),
        "int8_linear_quantize ", m, "x", k, " -> ", n);
}

Tensor mxfp8_scaled_mm(const Tensor& a, const Tensor& a_scale_swizzled, const Tensor& weight,
                       const Tensor& weight_exponent, const OptTensor& bias, bool weight_scale_e8m0) {
  check_dims(a, 2, "mxfp8_scaled_mm");
  const c10::DeviceGuard guard(a.device());
  const int64_t m = a.size(0), k = a.size(1), n = weight.size(0);
  Tensor out = empty({m, n}, a, at::kBFloat16);
  check(fim_mxfp8_scaled_mm(ptr<const uint8_t>(a), m, k, ptr<const uint8_t>(a_scale_swizzled),
                            ptr<const uint8_t>(weight), n, ptr<const int8_t>(weight_exponent), weight_scale_e8m0,
                            ptr<const void>(bias), bias_code(bias), out.data_ptr(), stream_of(a)),
        "mxfp8_scaled_mm ", m, "x", k, " -> ", n);
  return out;
}

Tensor im2col_gather(const Tensor& x, FIM_GEO_PARAMS) {
  check_dims(x, 4, "im2col_gather");
  const c10::DeviceGuard guard(x.device());
  const Geometry g = FIM_GEO;
  const int64_t b = x.size(0), h = x.size(1), w = x.size(2), c = x.size(3);
  TORCH_CHECK(sh > 0 && sw > 0, "im2col_gather: strides must be positive");
  Tensor out = empty({b * g.ho(h) * g.wo(w), kh * kw * c}, x, at::kByte);
  check(fim_im2col_gather(ptr<const uint8_t>(x), b, h, w, c, FIM_GEO_ARGS(g), ptr<uint8_t>(out), stream_of(x)),
        "im2col_gather");
  return out;
}

Tensor refiner_mlp(int64_t kind, int64_t semantics, const Tensor& x, const Tensor& x_scale, const Tensor& w1,
                   const Tensor& w1_scale, const OptTensor& b1, const Tensor& h_scale, const Tensor& w2,
                   const Tensor& w2_scale, const OptTensor& b2, const OptTensor& residual) {
  check_dims(x, 2, "refiner_mlp");
  const c10::DeviceGuard guard(x.device());
  const int64_t rows = x.size(0), c = x.size(1), h = w1.size(0);
  Tensor out = empty({rows, w2.size(0)}, x, at::kBFloat16);
  check(fim_refiner_mlp((int)kind, (int)semantics, ptr<const uint8_t>(x), rows, c, h, x_scale.data_ptr(),
                        ptr<const uint8_t>(w1), w1_scale.data_ptr(), ptr<const void>(b1), bias_code(b1),
                        h_scale.data_ptr(), ptr<const uint8_t>(w2), w2_scale.data_ptr(), ptr<const void>(b2),
                        bias_code(b2), ptr<const uint16_t>(residual), ptr<uint16_t>(out), stream_of(x)),
        "refiner_mlp ", rows, "x", c);
  return out;
}

constexpr int DW_MX_DYNAMIC = 0, DW_INT8 = 1, DW_BF16 = 2, DW_MX_STATIC = 3;

Tensor depthwise5x5(const Tensor& x, const Tensor& weight, const Tensor& bias, int64_t act, int64_t mode,
                    const OptTensor& scale, const OptTensor& exponent) {
  check_dims(x, 4, "depthwise5x5");
  const c10::DeviceGuard guard(x.device());
  TORCH_CHECK(mode == DW_INT8 || mode == DW_BF16 || mode == DW_MX_STATIC, "depthwise5x5: no output mode ", mode);
  const int64_t b = x.size(0), h = x.size(1), w = x.size(2), c = x.size(3);
  Tensor out = empty({b * h * w, c}, x, mode == DW_INT8 ? at::kChar : mode == DW_BF16 ? at::kBFloat16 : at::kByte);
  check(fim_depthwise5x5(ptr<const uint16_t>(x), b, h, w, c, ptr<const uint16_t>(weight), bias.data_ptr(),
                         bias_code(bias), (int)act, (int)mode, ptr<const float>(scale), ptr<const int8_t>(exponent),
                         out.data_ptr(), nullptr, nullptr, stream_of(x)),
        "depthwise5x5 ", x.sizes());
  return out;
}

std::tuple<Tensor, Tensor> depthwise5x5_mx_dynamic(const Tensor& x, const Tensor& weight, const Tensor& bias) {
  check_dims(x, 4, "depthwise5x5_mx_dynamic");
  const c10::DeviceGuard guard(x.device());
  const int64_t b = x.size(0), h = x.size(1), w = x.size(2), c = x.size(3), rows = b * h * w;
  Tensor out = empty({rows, c}, x, at::kByte), swz = swizzled_scales(rows, c / BLOCK, x);
  check(fim_depthwise5x5(ptr<const uint16_t>(x), b, h, w, c, ptr<const uint16_t>(weight), bias.data_ptr(),
                         bias_code(bias), 0, DW_MX_DYNAMIC, nullptr, nullptr, out.data_ptr(), nullptr,
                         ptr<uint8_t>(swz), stream_of(x)),
        "depthwise5x5 ", x.sizes());
  return {out, swz};
}

Tensor depthwise5x5_relu_pointwise_mxfp8(const Tensor& x, const Tensor& dw_weight, const Tensor& dw_bias,
                                         const Tensor& pw_weight, const Tensor& pw_e8m0, const OptTensor& pw_bias) {
  check_dims(x, 4, "depthwise5x5_relu_pointwise_mxfp8");
  const c10::DeviceGuard guard(x.device());
  const int64_t b = x.size(0), h = x.size(1), w = x.size(2), c = x.size(3), n = pw_weight.size(0);
  Tensor out = empty({b, h, w, n}, x, at::kBFloat16);
  check(fim_depthwise5x5_relu_pointwise_mxfp8(ptr<const uint16_t>(x), b, h, w, c, ptr<const uint16_t>(dw_weight),
                                              dw_bias.data_ptr(), bias_code(dw_bias), ptr<const uint8_t>(pw_weight), n,
                                              ptr<const uint8_t>(pw_e8m0), ptr<const void>(pw_bias), bias_code(pw_bias),
                                              ptr<uint16_t>(out), stream_of(x)),
        "depthwise5x5_relu_pointwise_mxfp8 ", x.sizes());
  return out;
}

Tensor depthwise5x5_relu_pointwise_int8(const Tensor& x, const Tensor& dw_weight, const Tensor& dw_bias,
                                        const Tensor& scale, const Tensor& pw_weight, const Tensor& pw_wscale,
                                        const OptTensor& pw_bias) {
  check_dims(x, 4, "depthwise5x5_relu_pointwise_int8");
  const c10::DeviceGuard guard(x.device());
  const int64_t b = x.size(0), h = x.size(1), w = x.size(2), c = x.size(3), n = pw_weight.size(0);
  Tensor out = empty({b, h, w, n}, x, at::kBFloat16);
  check(fim_depthwise5x5_relu_pointwise_int8(ptr<const uint16_t>(x), b, h, w, c, ptr<const uint16_t>(dw_weight),
                                             dw_bias.data_ptr(), bias_code(dw_bias), ptr<const float>(scale),
                                             ptr<const int8_t>(pw_weight), n, ptr<const float>(pw_wscale),
                                             ptr<const void>(pw_bias), bias_code(pw_bias), ptr<uint16_t>(out),
                                             stream_of(x)),
        "depthwise5x5_relu_pointwise_int8 ", x.sizes());
  return out;
}

Tensor conv3x3_small_cin_quantize_int8(const Tensor& x, const Tensor& packed, const Tensor& bias, const Tensor& scale) {
  check_dims(x, 4, "conv2d_small_cin_quantize_int8");
  const c10::DeviceGuard guard(x.device());
  const int64_t b = x.size(0), cin = x.size(1), h = x.size(2), w = x.size(3), cout = packed.size(0);
  Tensor out = empty({b, h, w, cout}, x, at::kChar);
  check(fim_conv3x3_small_cin_quantize_int8(ptr<const uint16_t>(x), b, cin, h, w, ptr<const uint16_t>(packed), cout,
                                            bias.data_ptr(), bias_code(bias), ptr<const float>(scale),
                                            ptr<int8_t>(out), stream_of(x)),
        "conv2d_small_cin_quantize_int8 ", x.sizes(), " -> ", cout);
  return out;
}

Tensor bias_relu_quantize_int8(const Tensor& raw, const Tensor& bias, const Tensor& scale) {
  check_dims(raw, 4, "bias_relu_quantize_int8");
  const c10::DeviceGuard guard(raw.device());
  const int64_t b = raw.size(0), c = raw.size(1), h = raw.size(2), w = raw.size(3);
  Tensor out = empty({b, h, w, c}, raw, at::kChar);
  check(fim_bias_relu_quantize_int8(ptr<const uint16_t>(raw), b, c, h, w, bias.data_ptr(), bias_code(bias),
                                    ptr<const float>(scale), ptr<int8_t>(out), stream_of(raw)),
        "bias_relu_quantize_int8 ", raw.sizes());
  return out;
}

Tensor pointwise_bf16(const Tensor& x, const Tensor& weight, const OptTensor& bias) {
  check_dims(x, 2, "pointwise_bf16");
  const c10::DeviceGuard guard(x.device());
  const int64_t m = x.size(0), k = x.size(1), n = weight.size(0);
  Tensor out = empty({m, n}, x, at::kBFloat16);
  check(fim_pointwise_bf16(ptr<const uint16_t>(x), m, k, ptr<const uint16_t>(weight), n, ptr<const void>(bias),
                           bias_code(bias), ptr<uint16_t>(out), stream_of(x)),
        "pointwise_bf16 ", m, "x", k, "x", n);
  return out;
}

}  // namespace

#define FIM_GEO_SCHEMA "SymInt kh, SymInt kw, SymInt sh, SymInt sw, SymInt ph, SymInt pw, SymInt dh, SymInt dw"

// name, schema, function: one row per operator
#define FIM_OPS(X)                                                                                                     \
  X(quantize_mxfp8, "(Tensor value, Tensor exponent, SymInt padded) -> Tensor")                                        \
  X(gelu_quantize_mxfp8,                                                                                               \
    "(Tensor value, Tensor exponent, SymInt padded, Tensor? input_bias, bool tanh=False) -> Tensor")                   \
  X(quantize_int8, "(Tensor value, Tensor scale, Tensor? channel_scale) -> Tensor")                                    \
  X(gelu_quantize_int8, "(Tensor value, Tensor scale, bool tanh=False) -> Tensor")                                     \
  X(quantize_mxfp8_dynamic, "(Tensor value, bool swizzled) -> (Tensor, Tensor)")                                       \
  X(quantize_int8_rows, "(Tensor value, bool reciprocal) -> (Tensor, Tensor)")                                         \
  X(calibrate_block32, "(Tensor matrix) -> Tensor")                                                                    \
  X(int8_conv2d, "(Tensor x, Tensor weight, Tensor a_scale, Tensor w_scale, Tensor? bias, " FIM_GEO_SCHEMA             \
                 ", bool relu, bool gelu, Tensor? residual, Tensor? out_scale) -> Tensor")                             \
  X(int8_conv2d_maxpool, "(Tensor x, Tensor weight, Tensor a_scale, Tensor w_scale, Tensor? bias, " FIM_GEO_SCHEMA     \
                         ", bool relu, Tensor out_scale) -> (Tensor, Tensor)")                                         \
  X(mxfp8_conv2d, "(Tensor x, Tensor channel_exponent, Tensor weight, Tensor weight_exponent, Tensor? bias, "          \
                  FIM_GEO_SCHEMA ", bool relu, bool gelu, Tensor? residual, Tensor? out_exponent) -> Tensor")          \
  X(int8_linear, "(Tensor a, Tensor weight, Tensor a_scale, Tensor w_scale, Tensor? bias, bool relu, bool gelu, "      \
                 "Tensor? residual) -> Tensor")                                                                        \
  X(int8_linear_quantize_, "(Tensor a, Tensor weight, Tensor a_scale, Tensor w_scale, Tensor? bias, "                  \
                           "Tensor out_scale, Tensor(a!) out) -> ()")                                                  \
  X(mxfp8_scaled_mm, "(Tensor a, Tensor a_scale_swizzled, Tensor weight, Tensor weight_exponent, Tensor? bias, "       \
                     "bool weight_scale_e8m0=False) -> Tensor")                                                        \
  X(im2col_gather, "(Tensor x, " FIM_GEO_SCHEMA ") -> Tensor")                                                         \
  X(refiner_mlp, "(SymInt kind, SymInt semantics, Tensor x, Tensor x_scale, Tensor w1, Tensor w1_scale, Tensor? b1, "  \
                 "Tensor h_scale, Tensor w2, Tensor w2_scale, Tensor? b2, Tensor? residual) -> Tensor")                \
  X(depthwise5x5, "(Tensor x, Tensor weight, Tensor bias, SymInt act, SymInt mode, Tensor? scale, Tensor? exponent) "  \
                  "-> Tensor")                                                                                         \
  X(depthwise5x5_mx_dynamic, "(Tensor x, Tensor weight, Tensor bias) -> (Tensor, Tensor)")                             \
  X(depthwise5x5_relu_pointwise_mxfp8, "(Tensor x, Tensor dw_weight, Tensor dw_bias, Tensor pw_weight, "               \
                                       "Tensor pw_e8m0, Tensor? pw_bias) -> Tensor")                                   \
  X(depthwise5x5_relu_pointwise_int8, "(Tensor x, Tensor dw_weight, Tensor dw_bias, Tensor scale, Tensor pw_weight, "  \
                                      "Tensor pw_wscale, Tensor? pw_bias) -> Tensor")                                  \
  X(conv3x3_small_cin_quantize_int8, "(Tensor x, Tensor packed, Tensor bias, Tensor scale) -> Tensor")                 \
  X(bias_relu_quantize_int8, "(Tensor raw, Tensor bias, Tensor scale) -> Tensor")                                      \
  X(pointwise_bf16, "(Tensor x, Tensor weight, Tensor? bias) -> Tensor")

TORCH_LIBRARY(flashim_amd, m) {
#define X(name, schema) m.def(#name schema, {at::Tag::pt2_compliant_tag});
  FIM_OPS(X)
#undef X
}

TORCH_LIBRARY_IMPL(flashim_amd, CUDA, m) {
#define X(name, schema) m.impl(#name, TORCH_FN(name));
  FIM_OPS(X)
#undef X
}

namespace {

// No derivative formulas. Reverse mode: the outputs of inputs that require a gradient carry a node that raises. Forward
// mode alone: the tangents of dual inputs stop here and the outputs have none (torch's own fallback for operators without
// formulas refuses every dual input).
void no_derivative(const c10::OperatorHandle& op, c10::DispatchKeySet keys, torch::jit::Stack* stack) {
  const std::string& name = op.schema().name();
  torch::autograd::variable_list inputs;  // that require a gradient
  if (at::GradMode::is_enabled()) {
    bool dual = false;
    for (const c10::IValue& arg : torch::jit::last(*stack, op.schema().arguments().size()))
      if (arg.isTensor()) {
        const Tensor& t = arg.toTensor();
        if (t.requires_grad()) inputs.push_back(t);
        dual = dual || torch::autograd::isFwGradDefined(t);
      }
    TORCH_CHECK_NOT_IMPLEMENTED(inputs.empty() || !dual, name,
                                ": no forward-mode derivative, and an input requires a gradient");
  }
  {
    at::AutoDispatchBelowAutograd guard;
    op.redispatchBoxed(keys & c10::after_autograd_keyset, stack);
  }
  if (inputs.empty()) return;
  std::shared_ptr<torch::autograd::Node> node(new torch::autograd::NotImplemented(name), torch::autograd::deleteNode);
  node->set_next_edges(torch::autograd::collect_next_edges(inputs));
  for (const c10::IValue& out : torch::jit::last(*stack, op.schema().returns().size()))
    if (out.isTensor() && torch::autograd::isDifferentiableType(out.toTensor().scalar_type()))
      torch::autograd::set_history(out.toTensor(), node);
}

// The version counter of the last argument, the tensor that is written, by which autograd finds a saved tensor that was
// overwritten since (torch's own fallback counts for returned tensors only).
void count_write_to_last(const c10::OperatorHandle& op, c10::DispatchKeySet keys, torch::jit::Stack* stack) {
  const Tensor out = stack->back().toTensor();
  {
    at::AutoDispatchBelowADInplaceOrView guard;
    op.redispatchBoxed(keys & c10::after_ADInplaceOrView_keyset, stack);
  }
  if (!out.is_inference()) torch::autograd::increment_version(out);
}

}  // namespace

TORCH_LIBRARY_IMPL(flashim_amd, Autograd, m) {
#define X(name, schema) m.impl(#name, torch::CppFunction::makeFromBoxedFunction<&no_derivative>());
  FIM_OPS(X)
#undef X
}

TORCH_LIBRARY_IMPL(flashim_amd, ADInplaceOrView, m) {
  m.impl("int8_linear_quantize_", torch::CppFunction::makeFromBoxedFunction<&count_write_to_last>());
}
