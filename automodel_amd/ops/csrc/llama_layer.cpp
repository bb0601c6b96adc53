// One decode step of a Llama decoder layer: its launches in a row, without a
// return to Python in between. A layer is 9 launches of 2 to 40 us for one
// sequence; issued one by one from modules the host was the bound: 4 layers of
// 4096 columns took 0.62 ms a step, and 0.45 this way.

#include <torch/library.h>
#include <ATen/ATen.h>

#include "ops_api.h"

namespace amd_ops {

namespace {

// a weight that the kernels take as it is: bf16, whole, aligned
bool plain(const at::Tensor& w, const at::Tensor& x, int64_t rows, int64_t cols) {
  return w.device() == x.device() && w.scalar_type() == at::kBFloat16 && w.is_contiguous() &&
         w.dim() == (cols ? 2 : 1) && w.size(0) == rows && (!cols || w.size(1) == cols) &&
         reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0;
}

}  // namespace

// x [B, 1, width] bf16; ws: input norm, middle norm, o, down, then q, k, v (or all in
// one), then gate, up (or both in one). -> {the layer's output}, or {} where the kernels
// do not take these tensors, and then nothing has been done.
std::vector<at::Tensor> llama_decode_layer(
    const at::Tensor& x, at::TensorList ws, const at::Tensor& cos, const at::Tensor& sin,
    at::Tensor k_cache, at::Tensor v_cache, int64_t pos, const std::optional<at::Tensor>& pos_dev,
    double scale, double eps_in, double eps_mid, int64_t heads, int64_t kv_heads, bool fused_qkv,
    bool fused_gate_up) {
  if (!(x.is_cuda() && x.dim() == 3 && x.size(1) == 1 && x.is_contiguous() &&
        x.scalar_type() == at::kBFloat16 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 &&
        (int64_t)ws.size() == 4 + (fused_qkv ? 1 : 3) + (fused_gate_up ? 1 : 2)))
    return {};
  const int64_t B = x.size(0), W = x.size(2);
  if (B < 1 || B > 32 || W < 8 || W % 8 || W > 16384) return {};
  if (k_cache.dim() != 4 || k_cache.size(0) != B || k_cache.size(2) != kv_heads) return {};
  const int64_t D = k_cache.size(3), nq = heads * D, nk = kv_heads * D;
  const int64_t I = ws.back().dim() == 2 ? ws.back().size(0) / (fused_gate_up ? 2 : 1) : 0;
  if (D % 8 || D > 256 || heads % kv_heads || I < 8 || I % 8) return {};
  if (!(k_cache.device() == x.device() && k_cache.scalar_type() == at::kBFloat16)) return {};
  for (const at::Tensor* t : {&cos, &sin})
    if (!(t->device() == x.device() && t->scalar_type() == at::kFloat && t->dim() == 2 &&
          t->is_contiguous() && t->size(0) >= 1 && t->size(1) == D))
      return {};
  const auto &w_o = ws[2], &w_down = ws[3];
  std::vector<at::Tensor> qkv, glu;
  if (!(plain(ws[0], x, W, 0) && plain(ws[1], x, W, 0) && plain(w_o, x, W, nq) &&
        plain(w_down, x, W, I)))
    return {};
  if (fused_qkv) {
    if (!plain(ws[4], x, nq + 2 * nk, W)) return {};
    qkv = {ws[4].narrow(0, 0, nq), ws[4].narrow(0, nq, nk), ws[4].narrow(0, nq + nk, nk)};
  } else {
    if (!(plain(ws[4], x, nq, W) && plain(ws[5], x, nk, W) && plain(ws[6], x, nk, W))) return {};
    qkv = {ws[4], ws[5], ws[6]};
  }
  if (fused_gate_up) {
    if (!plain(ws.back(), x, 2 * I, W)) return {};
    glu = {ws.back().narrow(0, 0, I), ws.back().narrow(0, I, I)};
  } else {
    glu = {ws[ws.size() - 2], ws.back()};
    if (!(plain(glu[0], x, I, W) && plain(glu[1], x, I, W))) return {};
  }

  const auto rows = x.view({B, W});
  const auto h = std::get<0>(rms_norm_fwd(rows, ws[0], eps_in));
  const auto p = decode_rows(h, qkv);
  const auto [q, k] = rope_fwd(p[0].view({B, 1, heads, D}), p[1].view({B, 1, kv_heads, D}), cos,
                               sin, false);
  const auto o = kv_decode_attn(q, k, p[2].view({B, 1, kv_heads, D}), k_cache, v_cache, pos,
                                pos_dev, scale);
  const auto y = decode_rows(o.view({B, nq}), w_o);
  const auto [sum, h2, unused] = add_rms_norm_fwd(rows, y[0], ws[1], eps_mid);
  const auto act = decode_rows(h2, glu, true);
  return {decode_rows(act[0], w_down, false, false, sum)[0].view({B, 1, W})};
}

}  // namespace amd_ops
