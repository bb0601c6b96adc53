// y = x w^T as one node of autograd, for small layers: forward and backward are calls of some 5 us on the host, where
// a function of Python's is 20 each way and the library's products 28 each. The products are linear_small.hip's where
// these are the faster ones, else the library's.

#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <ATen/ATen.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include "ops_api.h"

namespace amd_ops {

namespace {

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Products of up to so many. Time of the kernels over the library's, captured, 5000 shapes of 1 to 8000 rows
// (profiles/sweep_linear_small.csv): nt from 17 rows on 0.3 to 1.6, 0.90 in the mean, above 1.05 for a quarter of them (512 rows and
// more, 2^31 products and more: 1.02 and half of them); nn 0.2 to 1.5 (0.76); tn 0.12 to 1.7 (0.65). Beyond, nt and nn 1.2, tn 0.8.
// The library's take another 24 us of the host, which a captured step does not see.
constexpr int64_t MOST = 1l << 32, MOST_TN = 1l << 33;

// what the kernels read as it is: memory to point to, and nothing between it and the tensor
bool plain(const at::Tensor& t) {
  using c10::DispatchKey;
  static const c10::DispatchKeySet followers({DispatchKey::Python, DispatchKey::FuncTorchBatched, DispatchKey::Batched,
                                              DispatchKey::FuncTorchGradWrapper, DispatchKey::Functionalize,
                                              DispatchKey::Conjugate, DispatchKey::Negative, DispatchKey::ZeroTensor});
  return t.is_cuda() && t.scalar_type() == at::kBFloat16 && !t.key_set().has_any(followers) && t.is_contiguous() &&
         reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

// Whether something besides autograd follows the operations: a dispatch mode (maybe around the backward alone), a
// transform, forward-mode derivatives, a trace. It sees into torch's operations but not into the kernels.
bool followed() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || torch::autograd::ForwardADLevel::try_get_by_idx(0) ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) || torch::jit::tracer::isTracing();
}

bool takes(const at::Tensor& a, const at::Tensor& b, int64_t T, int64_t N, int64_t K, int64_t most) {
  return !followed() && small_takes(T, N, K) && T * N * K < most && plain(a) && plain(b) && a.device() == b.device();
}

at::Tensor forward_of(const at::Tensor& x, const at::Tensor& w) {
  const int64_t N = w.size(0), K = w.size(1), T = K ? x.numel() / K : 0;
  if (!takes(x, w, T, N, K, MOST)) return at::linear(x, w);
  auto shape = x.sizes().vec();
  shape.back() = N;
  return small_nt(x.view({T, K}), w).view(shape);
}

struct SmallLinear : torch::autograd::Function<SmallLinear> {
  static at::Tensor forward(AutogradContext* ctx, const at::Tensor& x, const at::Tensor& w) {
    ctx->save_for_backward({w.requires_grad() ? x : at::Tensor(), x.requires_grad() ? w : at::Tensor()});
    ctx->saved_data["shape"] = x.sizes();
    return forward_of(x, w);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const auto saved = ctx->get_saved_variables();
    const auto &x = saved[0], &w = saved[1];
    const auto shape = ctx->saved_data["shape"].toIntVector();
    if (!grads[0].defined()) return {at::Tensor(), at::Tensor()};
    // recorded itself, or followed: torch's own operations
    const bool recorded = at::GradMode::is_enabled();
    auto g = grads[0].reshape({-1, grads[0].size(-1)});
    if (!recorded) g = g.contiguous();
    const int64_t T = g.size(0), N = g.size(1), K = shape.back();
    at::Tensor dx, dw;
    if (w.defined() && ctx->needs_input_grad(0))
      dx = (!recorded && takes(g, w, T, N, K, MOST) ? small_nn(g, w) : at::matmul(g, w)).view(shape);
    if (x.defined() && ctx->needs_input_grad(1)) {
      const auto x2 = x.reshape({-1, K});
      dw = !recorded && takes(g, x2, T, N, K, MOST_TN) ? small_tn(g, x2) : at::matmul(g.t(), x2);
    }
    return {dx, dw};
  }
};

}  // namespace

at::Tensor linear_small(const at::Tensor& x, const at::Tensor& w) {
  if (at::GradMode::is_enabled() && (x.requires_grad() || w.requires_grad())) return SmallLinear::apply(x, w);
  return forward_of(x, w);
}

}  // namespace amd_ops
