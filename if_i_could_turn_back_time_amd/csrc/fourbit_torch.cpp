// The packed linear layer's call path from torch: one native call per forward (and per activation
// gradient) instead of a dozen Python, ctypes and dispatcher steps.  It launches the kernels that
// linear.py's packed_linear launches, on x converted as there, and takes workspaces from the
// allocator; what it does not recognise (another dtype, a refused shape, a wrapped tensor or one
// with a forward-mode tangent, a bias that is no vector, an active dispatch mode) it leaves to
// packed_linear by returning None.  A decode call of a 4096^2 layer takes 5 us on the GPU and took
// 22 us of host time through Python.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/utils/pybind.h>

#include <algorithm>
#include <optional>
#include <stdexcept>

#include "fourbit.h"

namespace py = pybind11;

namespace {

constexpr int64_t kMaxGemvBatch = 16;
constexpr int64_t kMaxGemmK = 1 << 22;  // fb_gemm's limits
constexpr int64_t kMaxGemmRows = 1 << 24;
constexpr int64_t kMaxRotatedValues = 1 << 29;  // of x, rotated at once: a copy of 1 GiB
// Rows of grad_y at once: bounds fb_grad_x's 16-bit terms of them, and each pass's decode of W
// is under 1% of its products.
constexpr int64_t kGradRows = 8192;

void check(int code) {
  if (code != FB_OK) throw std::runtime_error(fb_strerror(code));
}

int dtype_code(at::ScalarType t) {
  return t == at::kHalf ? FB_DT_F16 : t == at::kBFloat16 ? FB_DT_BF16 : t == at::kFloat ? FB_DT_F32 : -1;
}

// A plain dense GPU tensor whose memory this code may read: no functorch wrapper, fake or
// functional tensor, and no forward-mode tangent, which only torch operations carry on.
bool plain(const at::Tensor& t) {
  const auto ks = t.key_set();
  return !t._fw_grad(0).defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() &&
         !ks.has(c10::DispatchKey::Python) && !ks.has(c10::DispatchKey::Functionalize) &&
         !ks.has(c10::DispatchKey::FuncTorchBatched) &&
         !ks.has(c10::DispatchKey::FuncTorchGradWrapper) && !t.is_neg() && !t.is_conj();
}

// Whether somebody watches the operators.
bool watched() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer) ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

void* stream_of(const at::Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

at::Tensor scratch(size_t bytes, const at::Tensor& like) {
  return at::empty({(int64_t)bytes}, like.options().dtype(at::kByte));
}

void* ptr_or_null(const at::Tensor& t, size_t bytes) { return bytes ? t.data_ptr() : nullptr; }

// F.linear(x, W, bias) for a packed W, no gradients; None where packed_linear has to decide.
std::optional<at::Tensor> linear_forward(const at::Tensor& x, const at::Tensor& wdev, int64_t N,
                                         int64_t K, int64_t fmt, int64_t fwht_block, bool f16_exact,
                                         bool fp4_mfma, const std::optional<at::Tensor>& bias,
                                         bool bf16_exact) {
  if (watched() || !plain(x) || !plain(wdev) || x.device() != wdev.device() || x.dim() < 1 ||
      x.size(-1) != K || K < 1 || x.numel() == 0)
    return std::nullopt;
  // a bias of more dimensions broadcasts against the [M, N] product, not against y's shape
  if (bias && (!plain(*bias) || bias->device() != x.device() || bias->dim() > 1))
    return std::nullopt;
  const int xdt = dtype_code(x.scalar_type());
  if (xdt < 0) return std::nullopt;
  const bool e2m1 = fmt == FB_FMT_E2M1;
  if (fp4_mfma && (!e2m1 || fwht_block)) return std::nullopt;
  int kdt = xdt;  // the kernels' activation dtype
  if (!e2m1 || fwht_block)
    kdt = FB_DT_F16;
  else if (fp4_mfma || xdt == FB_DT_F32)
    kdt = FB_DT_BF16;
  if (e2m1 && kdt == FB_DT_F16 && !f16_exact) return std::nullopt;
  const int64_t kp = (K + 127) / 128 * 128, M = x.numel() / K;
  if (M > INT32_MAX || (M > kMaxGemvBatch && kp > kMaxGemmK)) return std::nullopt;
  // the GEMM decodes to bf16; the split of more than one GEMV batch is linear.py's
  if (M > kMaxGemvBatch && fp4_mfma && !bf16_exact) return std::nullopt;

  fb_shape_t s{};
  s.N = (int32_t)N;
  s.K = (int32_t)kp;
  s.B = (int32_t)std::min(M, fwht_block ? std::min(kMaxGemmRows, kMaxRotatedValues / kp / 16 * 16)
                                       : kMaxGemmRows);  // rows of a call
  s.group = e2m1 ? 32 : 128;
  s.fmt = (int32_t)fmt;
  s.fwht_block = (int32_t)fwht_block;
  s.x_dtype = kdt;
  s.y_dtype = xdt;
  if ((size_t)wdev.numel() < fb_device_bytes(&s) || !fb_device_bytes(&s)) return std::nullopt;

  c10::DeviceGuard guard(x.device());
  void* const stream = stream_of(x);
  const at::Tensor xc = x.is_contiguous() ? x : x.contiguous();
  at::Tensor xk = xc;
  if (kdt != xdt || kp != K) {
    xk = at::empty({M, kp}, x.options().dtype(kdt == FB_DT_F16 ? at::kHalf : at::kBFloat16));
    check(fb_cast_rows(xc.data_ptr(), xdt, (int32_t)M, (int32_t)K, xk.data_ptr(), kdt,
                       (int32_t)kp, stream));
  }
  if (reinterpret_cast<uintptr_t>(xk.data_ptr()) & 15u) return std::nullopt;
  // a bias that is a plain vector is added by the GEMM, or by one small kernel
  const bool vector_bias = bias && bias->dim() == 1 && bias->size(0) == N &&
                           bias->is_contiguous() && dtype_code(bias->scalar_type()) >= 0;
  const int bdt = vector_bias ? dtype_code(bias->scalar_type()) : 0;
  auto sizes = x.sizes().vec();
  sizes.back() = N;
  at::Tensor y = at::empty(sizes, x.options());
  if (M > kMaxGemvBatch) {
    const int64_t step = s.B;
    for (int64_t r = 0; r < M; r += step) {
      s.B = (int32_t)std::min(step, M - r);
      const size_t need = fb_gemm_workspace_bytes(&s);
      const at::Tensor ws = need ? scratch(need, x) : at::Tensor();
      check(fb_gemm(wdev.data_ptr(), static_cast<const char*>(xk.data_ptr()) + r * kp * 2,
                    static_cast<char*>(y.data_ptr()) + r * N * y.element_size(), &s,
                    vector_bias ? bias->data_ptr() : nullptr, bdt, ptr_or_null(ws, need), need,
                    stream));
    }
    if (vector_bias) return y;
  } else if (fp4_mfma) {
    const size_t need = fb_mx_workspace_bytes(&s);
    if (!need) return std::nullopt;
    const at::Tensor ws = scratch(need, x);
    check(fb_gemv_mx(wdev.data_ptr(), xk.data_ptr(), y.data_ptr(), &s, ws.data_ptr(), need,
                     stream));
  } else {
    const size_t need = fb_workspace_bytes(&s);
    const at::Tensor ws = need ? scratch(need, x) : at::Tensor();
    check(fb_gemv(wdev.data_ptr(), xk.data_ptr(), y.data_ptr(), &s, ptr_or_null(ws, need), need,
                  stream));
  }
  if (vector_bias)
    check(fb_add_bias(y.data_ptr(), xdt, (int32_t)M, (int32_t)N, bias->data_ptr(), bdt, stream));
  else if (bias)
    y.add_(bias->scalar_type() == y.scalar_type() ? *bias : bias->to(y.scalar_type()));
  return y;
}

// gx[M, K] = (gy . W) H for gy [M, N], in xdtype; None where the caller has to decide.
std::optional<at::Tensor> linear_grad_x(const at::Tensor& gy, const at::Tensor& wdev, int64_t N,
                                        int64_t K, int64_t fmt, int64_t fwht_block, bool f16_exact,
                                        at::ScalarType xt) {
  const int gdt = dtype_code(gy.scalar_type()), xdt = dtype_code(xt);
  const int64_t kp = (K + 127) / 128 * 128;
  if (watched() || !plain(gy) || !plain(wdev) || gy.device() != wdev.device() || gy.dim() != 2 ||
      gy.size(1) != N || gdt < 0 || xdt < 0 || gy.numel() == 0)
    return std::nullopt;
  fb_shape_t s{};
  s.N = (int32_t)N;
  s.K = (int32_t)kp;
  s.B = (int32_t)std::min(gy.size(0), kGradRows);
  s.group = fmt == FB_FMT_E2M1 ? 32 : 128;
  s.fmt = (int32_t)fmt;
  s.fwht_block = (int32_t)fwht_block;
  s.x_dtype = FB_DT_F16;
  s.y_dtype = gdt;
  if (!fb_grad_x_workspace_bytes(&s, f16_exact) || (size_t)wdev.numel() < fb_device_bytes(&s))
    return std::nullopt;
  c10::DeviceGuard guard(gy.device());
  const at::Tensor g = gy.contiguous();
  at::Tensor gx = at::empty({gy.size(0), kp}, gy.options().dtype(xt));
  for (int64_t r = 0; r < gy.size(0); r += kGradRows) {
    s.B = (int32_t)std::min(gy.size(0) - r, kGradRows);
    const size_t need = fb_grad_x_workspace_bytes(&s, f16_exact);
    const at::Tensor ws = scratch(need, gy);
    check(fb_grad_x(wdev.data_ptr(), static_cast<const char*>(g.data_ptr()) + r * N * g.element_size(),
                    static_cast<char*>(gx.data_ptr()) + r * kp * gx.element_size(), &s, xdt,
                    f16_exact, ws.data_ptr(), need, stream_of(gy)));
  }
  return kp == K ? gx : gx.narrow(1, 0, K).contiguous();
}

// The bias gradient: gy's column sums in bdtype; None where the caller has to decide.
std::optional<at::Tensor> linear_grad_bias(const at::Tensor& gy, at::ScalarType bt) {
  const int gdt = dtype_code(gy.scalar_type()), bdt = dtype_code(bt);
  if (watched() || !plain(gy) || gy.dim() != 2 || gdt < 0 || bdt < 0 || gy.numel() == 0 ||
      gy.size(0) > INT32_MAX || gy.size(1) > INT32_MAX)
    return std::nullopt;
  c10::DeviceGuard guard(gy.device());
  const at::Tensor g = gy.contiguous();
  at::Tensor gb = at::empty({gy.size(1)}, gy.options().dtype(bt));
  const int32_t M = (int32_t)gy.size(0), N = (int32_t)gy.size(1);
  const size_t need = fb_grad_bias_workspace_bytes(M, N);
  const at::Tensor ws = need ? scratch(need, gy) : at::Tensor();
  check(fb_grad_bias_ws(g.data_ptr(), gdt, M, N, gb.data_ptr(), bdt, ptr_or_null(ws, need), need,
                        stream_of(gy)));
  return gb;
}

// y, which holds bias [N] already, as a function of it.  A node of its own, and one that knows
// which gradients a backward pass asks for: autograd runs a Python function's whole backward for
// any one of its inputs, so as an input of linear.py's _PackedLinearFn the bias's gradient alone
// would compute gx too.
struct AddedBias : torch::autograd::Function<AddedBias> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& y,
                            const at::Tensor& bias) {
    ctx->mark_dirty({y});
    ctx->saved_data["dtype"] = bias.scalar_type();
    return y;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const at::Tensor& gy = grads[0];
    at::Tensor gb;
    if (ctx->needs_input_grad(1)) {
      const at::ScalarType bt = ctx->saved_data["dtype"].toScalarType();
      std::optional<at::Tensor> sums;
      if (!at::GradMode::is_enabled()) sums = linear_grad_bias(gy, bt);
      gb = sums ? *sums : gy.sum(0).to(bt);
    }
    return {gy, gb};
  }
};

at::Tensor added_bias(const at::Tensor& y, const at::Tensor& bias) {
  return AddedBias::apply(y, bias);
}

}  // namespace

PYBIND11_MODULE(_fourbit_torch, m) {
  m.def("linear_forward", &linear_forward);
  m.def("linear_grad_x", &linear_grad_x);
  m.def("linear_grad_bias", &linear_grad_bias);
  m.def("added_bias", &added_bias);
}
