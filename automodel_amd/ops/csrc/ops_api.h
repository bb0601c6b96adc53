// Declarations of all HIP op entry points (implemented in the sibling .hip TUs).
#pragma once

#include <ATen/ATen.h>
#include <tuple>

namespace amd_ops {

std::tuple<at::Tensor, at::Tensor> rms_norm_fwd(const at::Tensor& x, const at::Tensor& w,
                                                double eps);
std::tuple<at::Tensor, at::Tensor, at::Tensor> add_rms_norm_fwd(const at::Tensor& x,
                                                                const at::Tensor& delta,
                                                                const at::Tensor& w, double eps);
std::tuple<at::Tensor, at::Tensor> rms_norm_bwd(const at::Tensor& dy, const at::Tensor& x,
                                                const at::Tensor& w, const at::Tensor& invrms,
                                                const std::optional<at::Tensor>& dres = std::nullopt,
                                                bool want_dw = true);

std::tuple<at::Tensor, at::Tensor> rope_fwd(const at::Tensor& q, const at::Tensor& k,
                                            const at::Tensor& cosb, const at::Tensor& sinb,
                                            bool backward);

std::tuple<at::Tensor, at::Tensor, at::Tensor> rope_split(const at::Tensor& qkv, const at::Tensor& cosb,
                                                          const at::Tensor& sinb, int64_t Hq, int64_t Hk);
std::tuple<at::Tensor, at::Tensor, at::Tensor> token_rows(const at::Tensor& ids, const at::Tensor& table,
                                                          const at::Tensor& pos, const at::Tensor& cos,
                                                          const at::Tensor& sin);
at::Tensor rope_join(const at::Tensor& dq, const at::Tensor& dk, const at::Tensor& dv, const at::Tensor& cosb,
                     const at::Tensor& sinb);

at::Tensor swiglu_fwd(const at::Tensor& g, const at::Tensor& u);
at::Tensor swiglu_cat_fwd(const at::Tensor& gu);
at::Tensor swiglu_cat_bwd(const at::Tensor& dy, const at::Tensor& gu);
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> swiglu_rows_bwd(const at::Tensor& dh, const at::Tensor& g,
                                                                           const at::Tensor& u, const at::Tensor& p,
                                                                           const at::Tensor& order);
std::tuple<at::Tensor, at::Tensor> swiglu_bwd(const at::Tensor& dy, const at::Tensor& g,
                                              const at::Tensor& u);

void adamw_steps(at::TensorList params, at::TensorList grads, at::TensorList masters,
                 at::TensorList ms, at::TensorList vs, at::IntArrayRef steps, double lr,
                 double beta1, double beta2, double eps, double weight_decay);
void adamw_step(at::Tensor param, at::Tensor grad, at::Tensor master, at::Tensor m,
                at::Tensor v, int64_t step, double lr, double beta1, double beta2,
                double eps, double weight_decay);

std::tuple<at::Tensor, at::Tensor> flash_attn_fwd(
    const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, double scale,
    bool causal, int64_t q_start,
    const std::optional<at::Tensor>& doc_start = std::nullopt,
    const std::optional<at::Tensor>& sink = std::nullopt);
// whether dK/dV and dQ of such a call have the kernels in a given order; docs: documents of a packed row,
// 0: rows of their own, -1: documents, but not known how many
std::tuple<bool, int64_t> flash_attn_bwd_dq(int64_t B, int64_t Sq, int64_t Skv, int64_t Hq, int64_t Hk, int64_t Dqk,
                                            int64_t Dv, bool causal, int64_t q_start);
int64_t flash_attn_bwd_parts(int64_t B, int64_t Sq, int64_t Skv, int64_t Hq, int64_t Hk, int64_t Dqk, int64_t Dv,
                             bool causal, int64_t q_start, int64_t docs);
std::tuple<bool, bool> flash_attn_bwd_ordered(int64_t B, int64_t Sq, int64_t Skv, int64_t Hq, int64_t Hk,
                                              int64_t Dqk, int64_t Dv, bool causal, int64_t docs);
std::tuple<at::Tensor, at::Tensor, at::Tensor> flash_attn_bwd(
    const at::Tensor& dout, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
    const at::Tensor& o, const at::Tensor& lse, double scale, bool causal,
    int64_t q_start,
    const std::optional<at::Tensor>& doc_start = std::nullopt,
    const std::optional<at::Tensor>& doc_end = std::nullopt, int64_t docs = 0);

at::Tensor mfma_probe(const at::Tensor& a, const at::Tensor& b);
at::Tensor tr16_probe(const at::Tensor& pattern);

std::tuple<at::Tensor, at::Tensor> ce_fwd_logits(const at::Tensor& logits,
                                                 const at::Tensor& labels,
                                                 at::Tensor loss_sum);
void ce_bwd_logits(at::Tensor logits, const at::Tensor& labels, const at::Tensor& lse,
                   const at::Tensor& dloss, int64_t vocab_offset);
at::Tensor ce_grad_logits(const at::Tensor& logits, const at::Tensor& labels,
                          const at::Tensor& lse, const at::Tensor& dloss, int64_t vocab_offset);
std::tuple<at::Tensor, at::Tensor> ce_stats_logits(const at::Tensor& logits);

std::tuple<at::Tensor, at::Tensor> fused_ce_fwd(const at::Tensor& hidden,
                                                const at::Tensor& weight,
                                                const at::Tensor& labels);

std::tuple<at::Tensor, at::Tensor, at::Tensor> soft_ce_fwd(const at::Tensor& s,
                                                           const at::Tensor& t);
at::Tensor soft_ce_bwd(const at::Tensor& s, const at::Tensor& t,
                       const at::Tensor& lse_s, const at::Tensor& lse_t,
                       const at::Tensor& dloss);

at::Tensor nf4_dequant(const at::Tensor& packed, const at::Tensor& absmax,
                       int64_t block_size, int64_t rows, int64_t cols);
at::Tensor fp8_cast(const at::Tensor& x, const at::Tensor& scale, at::Tensor amax_out,
                    bool e5m2);
at::Tensor fp8_transpose(const at::Tensor& x8);
std::tuple<at::Tensor, at::Tensor> lora_apply(const std::optional<at::Tensor>& y, const at::Tensor& x,
                                              const at::Tensor& A, const at::Tensor& B, double scale);
std::tuple<at::Tensor, at::Tensor> lora_forward(const at::Tensor& y, const at::Tensor& x, const at::Tensor& A,
                                                const at::Tensor& B, double scale);
void lora_down(const at::Tensor& x, const at::Tensor& A, int64_t r, at::Tensor* t, at::Tensor* turned, double scale,
               double scale_turned);
std::tuple<at::Tensor, at::Tensor> lora_linear(const at::Tensor& x, const at::Tensor& w, const at::Tensor& A,
                                               const at::Tensor& B, double scale);
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> lora_grads(const at::Tensor& g, const at::Tensor& x,
                                                                      const at::Tensor& A, const at::Tensor& B,
                                                                      const at::Tensor& tt, double scale);
at::Tensor linear_dx_extra(const at::Tensor& g, const at::Tensor& w, const at::Tensor& t, const at::Tensor& a_t);
at::Tensor lora_fused_fwd(const at::Tensor& x, const at::Tensor& A,
                          const at::Tensor& B, double scale);
at::Tensor sgmv_fused_fwd(const at::Tensor& x, const at::Tensor& A,
                          const at::Tensor& B, const at::Tensor& scales,
                          const at::Tensor& offs, const at::Tensor& tile_map,
                          const std::optional<at::Tensor>& n_tiles = std::nullopt);

at::Tensor gemv_bf16(const at::Tensor& x, const at::Tensor& w,
                     const c10::optional<at::Tensor>& bias, bool relu2 = false,
                     bool out_f32 = false, int64_t group_n = 0);
at::Tensor device_ints(at::IntArrayRef values, at::Device device);
std::tuple<at::Tensor, at::Tensor> doc_bounds(const at::Tensor& cu, int64_t total);
at::Tensor kv_decode_attn(const at::Tensor& q, const at::Tensor& k_new, const at::Tensor& v_new,
                          at::Tensor k_cache, at::Tensor v_cache, int64_t pos,
                          const std::optional<at::Tensor>& pos_dev, double scale);
// sixteens of rows a wave of the kernel in a given order, for a forward without documents; 0: the other one
int64_t flash_attn_fwd_ordered(int64_t B, int64_t Sq, int64_t Skv, int64_t Hq, int64_t Hk, int64_t Dqk, int64_t Dv,
                               bool causal, int64_t q_start);
// rows of W a workgroup, slots of its rings and waves that 3 to 16 rows of x take (see gemv.hip)
std::tuple<int64_t, int64_t, int64_t> decode_rows_shape(at::IntArrayRef n, int64_t K, int64_t B, bool glu,
                                                        int64_t group_n);
at::Tensor gemm_skinny_bf16(const at::Tensor& x, const at::Tensor& w, bool relu2, bool out_f32,
                            int64_t group_n = 0);
std::vector<at::Tensor> decode_rows(const at::Tensor& x, at::TensorList ws, bool glu = false,
                                    bool relu2 = false,
                                    const std::optional<at::Tensor>& residual = std::nullopt);
bool decode_rows_makes(int64_t B, int64_t K, bool sum, int64_t n);
std::vector<at::Tensor> decode_rows_normed(const at::Tensor& x, const at::Tensor& norm, double eps,
                                           at::TensorList ws, bool glu = false);
std::vector<at::Tensor> decode_rows_rotated(const at::Tensor& x, const at::Tensor& norm, double eps,
                                            const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                            const at::Tensor& cos, const at::Tensor& sin);
std::vector<at::Tensor> decode_rows_summed(const at::Tensor& sum, const at::Tensor& y, const at::Tensor& post,
                                           double mult, const at::Tensor& norm, double eps, const at::Tensor& w);
// Kernels of latent_decode_layer, which has checked what they take (gemv.hip, latent_decode.hip, residual_norm.hip).
// Pointers without a type are to bf16.
void decode_rows_to(const void* x, const void* w, void* y, int64_t B, int64_t K, int64_t n, bool relu2);
void decode_rows_summed_to(const float* sum, const void* y, const void* post, double mult, const void* norm, double eps,
                           const void* w, void* out, float* sum_out, int64_t B, int64_t K, int64_t n);
bool latent_prep_plain(int64_t width, int64_t rank, int64_t dn, int64_t dr);
void latent_check_step(const at::Tensor& cos, const at::Tensor& sin, const at::Tensor& pos, const at::Tensor& slot,
                       const at::Tensor& cache, int64_t R, int64_t rank, int64_t dr);
void latent_prep_rows(const void* qkv, const void* w_uk, const void* w_norm, double eps, const at::Tensor& cos,
                      const at::Tensor& sin, const at::Tensor& pos, const at::Tensor& slot, const at::Tensor& cache,
                      void* q, int64_t R, int64_t heads, int64_t dn, int64_t dr, int64_t rank);
void latent_attn_rows(const void* q, const at::Tensor& cache, const at::Tensor& slot, const at::Tensor& pos,
                      float* part_o, float* part_ml, int64_t R, int64_t H, int64_t C, int64_t rank, double scale,
                      int64_t splits);
bool latent_combine_folds(int64_t R, int64_t S);
void latent_combine_rows(const float* part_o, const float* part_ml, const void* w_uv, float* o_lat, void* out,
                         int64_t R, int64_t H, int64_t S, int64_t n, int64_t rank, int64_t dv);
void residual_add_norm_to(const float* before, float* x, const void* y, const void* w_post, double mult, double eps,
                          const void* w_next, void* h, int64_t T, int64_t W);
std::vector<at::Tensor> llama_decode_layer(
    const at::Tensor& x, at::TensorList ws, const at::Tensor& cos, const at::Tensor& sin,
    at::Tensor k_cache, at::Tensor v_cache, int64_t pos, const std::optional<at::Tensor>& pos_dev,
    double scale, double eps_in, double eps_mid, int64_t heads, int64_t kv_heads, bool fused_qkv,
    bool fused_gate_up);
std::vector<at::Tensor> latent_decode_layer(
    at::Tensor x, const at::Tensor& h, at::TensorList ws, const std::optional<at::Tensor>& w_next,
    const at::Tensor& cos, const at::Tensor& sin, const at::Tensor& pos, const at::Tensor& slot,
    at::Tensor cache, double eps, double latent_eps, double mult, double scale, int64_t heads,
    int64_t dn, int64_t dr, int64_t splits);

std::tuple<at::Tensor, at::Tensor, at::Tensor> build_group_plan(
    const at::Tensor& counts, int64_t M, int64_t bm = 128);
at::Tensor grouped_gemm_nt(const at::Tensor& x, const at::Tensor& w,
                           const at::Tensor& offs, const at::Tensor& tile_map,
                           const std::optional<at::Tensor>& n_tiles = std::nullopt,
                           int64_t bm = 128);
at::Tensor grouped_gemm_nn(const at::Tensor& g, const at::Tensor& w,
                           const at::Tensor& offs, const at::Tensor& tile_map,
                           const std::optional<at::Tensor>& n_tiles = std::nullopt,
                           int64_t bm = 128);
int64_t grouped_gemm_cap(int64_t mode, int64_t M, int64_t E, int64_t N, int64_t K);
at::Tensor grouped_gemm_tn(const at::Tensor& g, const at::Tensor& x, const at::Tensor& offs, int64_t E);
at::Tensor small_nt(const at::Tensor& x, const at::Tensor& w);
at::Tensor small_nn(const at::Tensor& g, const at::Tensor& w);
at::Tensor small_tn(const at::Tensor& g, const at::Tensor& x);
bool small_takes(int64_t T, int64_t N, int64_t K);
std::tuple<int64_t, int64_t> small_cut(int64_t rows, int64_t cols, int64_t sum);
at::Tensor linear_small(const at::Tensor& x, const at::Tensor& w);
at::Tensor linear_y(const at::Tensor& x, const at::Tensor& w, bool relu2);
std::tuple<at::Tensor, at::Tensor, at::Tensor> grouped_glu(const at::Tensor& x, const at::Tensor& w, const at::Tensor& up,
                                                           const at::Tensor& offs, const at::Tensor& tile_map,
                                                           const std::optional<at::Tensor>& n_tiles, int64_t bm);
at::Tensor linear_glu(const at::Tensor& x, const at::Tensor& w, const at::Tensor& up);
std::vector<int64_t> linear_y_cut(int64_t T, int64_t N, int64_t K);
at::Tensor linear_dw(const at::Tensor& g, const at::Tensor& x);
std::vector<int64_t> linear_grad_cut(bool dw, int64_t T, int64_t N, int64_t K);
at::Tensor linear_dx(const at::Tensor& g, const at::Tensor& w);
at::Tensor grouped_gemm_nt_fp8(const at::Tensor& x8, const at::Tensor& w8,
                               const at::Tensor& offs, const at::Tensor& tile_map,
                               const at::Tensor& scale,
                               const std::optional<at::Tensor>& n_tiles = std::nullopt,
                               int64_t bm = 128);
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor> route_plan(
    const at::Tensor& indices, const at::Tensor& probs, int64_t E);
at::Tensor router_linear(const at::Tensor& x, const at::Tensor& w);
std::tuple<at::Tensor, at::Tensor> router_linear_bwd(const at::Tensor& d, const at::Tensor& x,
                                                     const at::Tensor& w, bool want_dx, bool want_dw);
at::Tensor route_topk(const at::Tensor& scores, int64_t K);
at::Tensor route_weights(const at::Tensor& scores, const at::Tensor& idx, bool norm, double scale, bool bf16_out);
at::Tensor route_weights_bwd(const at::Tensor& dprobs, const at::Tensor& scores, const at::Tensor& idx, bool softmax,
                             bool norm, double scale);
at::Tensor permute_rows(const at::Tensor& x, const at::Tensor& pos);
at::Tensor unpermute_sum(const at::Tensor& yp, const at::Tensor& pos);
at::Tensor expert_load(const at::Tensor& indices, int64_t E);
std::tuple<at::Tensor, at::Tensor> combine_bwd(const at::Tensor& g, const at::Tensor& y,
                                               const at::Tensor& src, const at::Tensor& order,
                                               const at::Tensor& probs);
at::Tensor grouped_gemm_nn2(const at::Tensor& g1, const at::Tensor& w1, const at::Tensor& g2,
                            const at::Tensor& w2, const at::Tensor& offs, const at::Tensor& tile_map,
                            const std::optional<at::Tensor>& n_tiles, int64_t bm);
at::Tensor unpermute_combine(const at::Tensor& yp, const at::Tensor& pos,
                             const at::Tensor& probs);

// --- inference: f32 residual stream (residual_norm.hip) ---
at::Tensor embed_rms_norm(const at::Tensor& ids, const at::Tensor& table, const at::Tensor& w,
                          double eps);
at::Tensor residual_rms_norm(const at::Tensor& x, const at::Tensor& w, double eps);
at::Tensor residual_add_norm(at::Tensor x, const at::Tensor& y, const at::Tensor& w_post,
                             double mult, double eps_post,
                             const std::optional<at::Tensor>& w_next, double eps_next);
at::Tensor concat_cast(const at::Tensor& a, const at::Tensor& b, bool to_bf16);
at::Tensor relu2_(at::Tensor x);

// --- inference: latent attention (latent_attn.hip, latent_decode.hip) ---
std::tuple<at::Tensor, at::Tensor, at::Tensor> latent_prep(
    const at::Tensor& qkv, const at::Tensor& w, double eps, const at::Tensor& cos,
    const at::Tensor& sin, const at::Tensor& pos, const std::optional<at::Tensor>& slot,
    const std::optional<at::Tensor>& cache, int64_t heads, int64_t dn, int64_t dr,
    int64_t head_pad, int64_t rows_pad);
std::tuple<at::Tensor, at::Tensor> latent_assemble(const at::Tensor& kv, const at::Tensor& kr,
                                                   int64_t heads, int64_t dn, int64_t dv,
                                                   int64_t k_pad, int64_t v_pad, int64_t n_tok);
at::Tensor attn_rows(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                     const at::Tensor& base, const at::Tensor& count, double scale, bool out_f32,
                     const std::optional<at::Tensor>& sink = std::nullopt);
at::Tensor latent_decode_prep(const at::Tensor& qkv, const at::Tensor& w_uk,
                              const at::Tensor& w_norm, double eps, const at::Tensor& cos,
                              const at::Tensor& sin, const at::Tensor& pos, const at::Tensor& slot,
                              at::Tensor cache, int64_t heads, int64_t dn, int64_t dr);
std::tuple<at::Tensor, at::Tensor> latent_decode_attn(const at::Tensor& q, const at::Tensor& cache,
                                                      const at::Tensor& slot, const at::Tensor& pos,
                                                      int64_t rank, int64_t rot, double scale,
                                                      int64_t splits);
at::Tensor latent_decode_combine(const at::Tensor& part_o,
                                 const std::optional<at::Tensor>& part_ml, const at::Tensor& w_uv,
                                 int64_t dv);

// --- inference: grouped attention, chunks, sinks (gqa_attn.hip) ---
std::tuple<at::Tensor, at::Tensor, at::Tensor> gqa_prep(
    const at::Tensor& proj, const at::Tensor& cos, const at::Tensor& sin, const at::Tensor& pos,
    const std::optional<at::Tensor>& slot, const std::optional<at::Tensor>& seq_end,
    const std::optional<at::Tensor>& cu_seqlens, const std::optional<at::Tensor>& k_cache,
    const std::optional<at::Tensor>& v_cache, int64_t chunk, int64_t heads, int64_t kv_heads,
    int64_t d, int64_t dv, int64_t head_pad, int64_t v_pad, int64_t rows_pad, bool decode);
at::Tensor gqa_decode_attn(const at::Tensor& q, const at::Tensor& k_cache,
                           const at::Tensor& v_cache, const at::Tensor& slot,
                           const at::Tensor& pos, const std::optional<at::Tensor>& sink,
                           int64_t chunk, int64_t dv, double scale, int64_t splits);

// --- inference: hyper-connections (hyper.hip) ---
std::tuple<at::Tensor, at::Tensor> hyper_embed(const at::Tensor& ids, const at::Tensor& table,
                                               double scale, const at::Tensor& w_in,
                                               const at::Tensor& w_norm, double eps);
at::Tensor hyper_step(at::Tensor x, const at::Tensor& y, const std::optional<at::Tensor>& y2,
                      const std::optional<at::Tensor>& w_y, const std::optional<at::Tensor>& w_y2,
                      const at::Tensor& w_mix, const at::Tensor& w_out,
                      const std::optional<at::Tensor>& w_in, const at::Tensor& w_norm, double eps,
                      bool keep);
at::Tensor clamped_glu(const at::Tensor& gu, double limit, double alpha);

// --- inference: linear recurrences (linear_scan.hip) ---
at::Tensor causal_conv_silu(const at::Tensor& x, const at::Tensor& w, const at::Tensor& bias,
                            const at::Tensor& pos, const std::optional<at::Tensor>& slot,
                            const std::optional<at::Tensor>& seq_end,
                            const std::optional<at::Tensor>& state);
at::Tensor token_shift(const at::Tensor& h, const at::Tensor& mu, const at::Tensor& pos,
                       const std::optional<at::Tensor>& slot,
                       const std::optional<at::Tensor>& seq_end,
                       const std::optional<at::Tensor>& state);
at::Tensor gated_group_norm(const at::Tensor& y, const at::Tensor& z, const at::Tensor& w,
                            int64_t groups, double eps, bool gate_first);
at::Tensor ssd_prompt(const at::Tensor& xbc, const at::Tensor& dt_in, const at::Tensor& dt_bias,
                      const at::Tensor& a_log, const at::Tensor& d_skip, const at::Tensor& cu,
                      const std::optional<at::Tensor>& slot,
                      const std::optional<at::Tensor>& state, int64_t groups, int64_t N,
                      int64_t max_len);
at::Tensor ssd_decode(const at::Tensor& xbc, const at::Tensor& dt_in, const at::Tensor& dt_bias,
                      const at::Tensor& a_log, const at::Tensor& d_skip, const at::Tensor& slot,
                      at::Tensor state, int64_t groups, int64_t N);
at::Tensor wkv_prompt(const at::Tensor& r, const at::Tensor& k, const at::Tensor& v,
                      at::Tensor low, const at::Tensor& w0, const at::Tensor& u,
                      const at::Tensor& cu, const std::optional<at::Tensor>& slot,
                      const std::optional<at::Tensor>& state, int64_t max_len);
at::Tensor wkv_decode(const at::Tensor& proj, const at::Tensor& w2, const at::Tensor& w0,
                      const at::Tensor& u, const at::Tensor& w_norm, double eps,
                      const at::Tensor& slot, at::Tensor state);

}  // namespace amd_ops
