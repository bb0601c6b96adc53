// One decode step of a layer with latent attention and a squared-ReLU feed-forward
// around a float32 residual: its launches in a row, without a return to Python in
// between. 9 launches of 2 to 10 us for one sequence; issued one by one from modules
// the host was the bound: 6 layer runs of 2048 columns took 0.58 ms a step, and 0.49
// this way.

#include <torch/library.h>
#include <ATen/ATen.h>

#include "ops_api.h"

namespace amd_ops {

// x [T, width] float32, updated in place; h [T, width] bf16, its normed form. ws: the
// projection to queries and latent, the latent's norm, the latent's up-projections, the
// output projection, the norm after; with a feed-forward also the norm before it, up,
// down, and the norm after it. w_next: the norm that makes the next layer's input.
// -> {that input, empty without w_next}, or {} where the kernels do not take these
// tensors, and then nothing has been done.
std::vector<at::Tensor> latent_decode_layer(
    at::Tensor x, const at::Tensor& h, at::TensorList ws, const std::optional<at::Tensor>& w_next,
    const at::Tensor& cos, const at::Tensor& sin, const at::Tensor& pos, const at::Tensor& slot,
    at::Tensor cache, double eps, double latent_eps, double mult, double scale, int64_t heads,
    int64_t dn, int64_t dr, int64_t splits) {
  const bool mlp = ws.size() == 9;
  if (!(ws.size() == 5 || mlp) || !h.is_cuda() || h.dim() != 2) return {};
  const int64_t T = h.size(0), W = h.size(1);
  if (T < 1 || T > 64 || W < 8 || W % 8 || !x.is_contiguous() || x.sizes() != h.sizes()) return {};
  if (x.scalar_type() != at::kFloat || x.device() != h.device()) return {};
  auto plain = [&](const at::Tensor& t, int64_t dim) {
    return t.device() == h.device() && t.scalar_type() == at::kBFloat16 && t.is_contiguous() &&
           t.dim() == dim && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  auto is = [&](const at::Tensor& t, int64_t n, int64_t k) {
    return plain(t, 2) && t.size(0) == n && t.size(1) == k;
  };
  auto norm = [&](const at::Tensor& t) { return plain(t, 1) && t.size(0) == W; };
  const auto &w_in = ws[0], &w_latent = ws[1], &w_kv_b = ws[2], &w_o = ws[3];
  if (!plain(h, 2) || !plain(w_latent, 1) || !plain(w_kv_b, 2) || !plain(w_o, 2)) return {};
  const int64_t rank = w_latent.size(0), dv = w_o.size(1) / heads;
  if (!(is(w_in, heads * (dn + dr) + rank + dr, W) && is(w_kv_b, heads * (dn + dv), rank) &&
        is(w_o, W, heads * dv) && w_o.size(1) % 8 == 0 && norm(ws[4])))
    return {};
  if (mlp && !(norm(ws[5]) && plain(ws[6], 2) && ws[6].size(0) % 8 == 0 &&
               is(ws[6], ws[6].size(0), W) && is(ws[7], W, ws[6].size(0)) && norm(ws[8])))
    return {};
  if (w_next && !norm(*w_next)) return {};

  const auto qkv = decode_rows(h, w_in)[0];
  const auto q = latent_decode_prep(qkv, w_kv_b.narrow(0, 0, heads * dn), w_latent, latent_eps, cos,
                                    sin, pos, slot, cache, heads, dn, dr);
  const auto [part, ml] = latent_decode_attn(q, cache, slot, pos, rank, dr, scale, splits);
  const auto o = latent_decode_combine(part, ml, w_kv_b.narrow(0, heads * dn, heads * dv), dv);
  const auto y = decode_rows(o, w_o)[0];
  if (!mlp) return {residual_add_norm(x, y, ws[4], mult, eps, w_next, eps)};
  const auto h2 = residual_add_norm(x, y, ws[4], mult, eps, ws[5], eps);
  const auto up = decode_rows(h2, ws[6], false, true)[0];
  const auto down = decode_rows(up, ws[7])[0];
  return {residual_add_norm(x, down, ws[8], mult, eps, w_next, eps)};
}

}  // namespace amd_ops
