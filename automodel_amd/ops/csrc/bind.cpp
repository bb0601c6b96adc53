// TORCH_LIBRARY registration for the amd_ops namespace.
// Loaded from python via torch.ops.load_library (automodel_amd/ops/_backend.py).
// The inference ops register in bind_decode.cpp, so that they can also be
// linked into a library of their own (ops/build.py --decode).

#include <torch/library.h>

#include "ops_api.h"

TORCH_LIBRARY(amd_ops, m) {
  m.def("rms_norm_fwd(Tensor x, Tensor w, float eps) -> (Tensor, Tensor)");
  m.impl("rms_norm_fwd", &amd_ops::rms_norm_fwd);
  m.def(
      "llama_decode_layer(Tensor x, Tensor[] ws, Tensor cos, Tensor sin, Tensor(a!) k_cache, "
      "Tensor(b!) v_cache, int pos, Tensor? pos_dev, float scale, float eps_in, float eps_mid, "
      "int heads, int kv_heads, bool fused_qkv, bool fused_gate_up) -> Tensor[]");
  m.impl("llama_decode_layer", &amd_ops::llama_decode_layer);
  m.def("add_rms_norm_fwd(Tensor x, Tensor delta, Tensor w, float eps) -> (Tensor, Tensor, Tensor)");
  m.impl("add_rms_norm_fwd", &amd_ops::add_rms_norm_fwd);
  m.def(
      "rms_norm_bwd(Tensor dy, Tensor x, Tensor w, Tensor invrms, Tensor? dres=None, "
      "bool want_dw=True) -> (Tensor, Tensor)");
  m.impl("rms_norm_bwd", &amd_ops::rms_norm_bwd);

  m.def("rope_fwd(Tensor q, Tensor k, Tensor cos, Tensor sin, bool backward) -> (Tensor, Tensor)");
  m.impl("rope_fwd", &amd_ops::rope_fwd);
  m.def("rope_split(Tensor qkv, Tensor cos, Tensor sin, int heads, int kv_heads) -> (Tensor, Tensor, Tensor)");
  m.impl("rope_split", &amd_ops::rope_split);
  m.def("token_rows(Tensor ids, Tensor table, Tensor pos, Tensor cos, Tensor sin) -> (Tensor, Tensor, Tensor)");
  m.impl("token_rows", &amd_ops::token_rows);
  m.def("rope_join(Tensor dq, Tensor dk, Tensor dv, Tensor cos, Tensor sin) -> Tensor");
  m.impl("rope_join", &amd_ops::rope_join);

  m.def("swiglu_fwd(Tensor g, Tensor u) -> Tensor");
  m.impl("swiglu_fwd", &amd_ops::swiglu_fwd);
  m.def("swiglu_rows_bwd(Tensor dh, Tensor g, Tensor u, Tensor p, Tensor order) -> (Tensor, Tensor, Tensor, Tensor)");
  m.impl("swiglu_rows_bwd", &amd_ops::swiglu_rows_bwd);
  m.def("swiglu_bwd(Tensor dy, Tensor g, Tensor u) -> (Tensor, Tensor)");
  m.impl("swiglu_bwd", &amd_ops::swiglu_bwd);
  m.def("swiglu_cat_fwd(Tensor gu) -> Tensor");
  m.impl("swiglu_cat_fwd", &amd_ops::swiglu_cat_fwd);
  m.def("swiglu_cat_bwd(Tensor dy, Tensor gu) -> Tensor");
  m.impl("swiglu_cat_bwd", &amd_ops::swiglu_cat_bwd);

  m.def(
      "adamw_step(Tensor(a!) param, Tensor grad, Tensor(b!) master, Tensor(c!) m, "
      "Tensor(d!) v, int step, float lr, float beta1, float beta2, float eps, "
      "float weight_decay) -> ()");
  m.impl("adamw_step", &amd_ops::adamw_step);
  m.def(
      "adamw_steps(Tensor(a!)[] params, Tensor[] grads, Tensor(b!)[] masters, Tensor(c!)[] ms, "
      "Tensor(d!)[] vs, int[] steps, float lr, float beta1, float beta2, float eps, "
      "float weight_decay) -> ()");
  m.impl("adamw_steps", &amd_ops::adamw_steps);

  m.def(
      "flash_attn_bwd(Tensor dout, Tensor q, Tensor k, Tensor v, Tensor o, Tensor lse, "
      "float scale, bool causal, int q_start=0, Tensor? doc_start=None, "
      "Tensor? doc_end=None, int docs=0) -> (Tensor, Tensor, Tensor)");
  m.impl("flash_attn_bwd", &amd_ops::flash_attn_bwd);
  m.def("flash_attn_bwd_parts(int B, int Sq, int Skv, int Hq, int Hk, int Dqk, int Dv, bool causal, int q_start, "
        "int docs) -> int");
  m.impl("flash_attn_bwd_parts", &amd_ops::flash_attn_bwd_parts);
  m.def("flash_attn_bwd_dq(int B, int Sq, int Skv, int Hq, int Hk, int Dqk, int Dv, bool causal, int q_start) -> (bool, int)");
  m.impl("flash_attn_bwd_dq", &amd_ops::flash_attn_bwd_dq);
  m.def("flash_attn_bwd_ordered(int B, int Sq, int Skv, int Hq, int Hk, int Dqk, int Dv, bool causal, "
        "int docs=0) -> (bool, bool)");
  m.impl("flash_attn_bwd_ordered", &amd_ops::flash_attn_bwd_ordered);

  m.def("mfma_probe(Tensor a, Tensor b) -> Tensor");
  m.impl("mfma_probe", &amd_ops::mfma_probe);
  m.def("tr16_probe(Tensor pattern) -> Tensor");
  m.impl("tr16_probe", &amd_ops::tr16_probe);

  m.def("ce_fwd_logits(Tensor logits, Tensor labels, Tensor(a!) loss_sum) -> (Tensor, Tensor)");
  m.impl("ce_fwd_logits", &amd_ops::ce_fwd_logits);
  m.def("ce_bwd_logits(Tensor(a!) logits, Tensor labels, Tensor lse, Tensor dloss, int vocab_offset=0) -> ()");
  m.impl("ce_bwd_logits", &amd_ops::ce_bwd_logits);
  m.def("ce_grad_logits(Tensor logits, Tensor labels, Tensor lse, Tensor dloss, int vocab_offset=0) -> Tensor");
  m.impl("ce_grad_logits", &amd_ops::ce_grad_logits);
  m.def("ce_stats_logits(Tensor logits) -> (Tensor, Tensor)");
  m.impl("ce_stats_logits", &amd_ops::ce_stats_logits);

  m.def("fused_ce_fwd(Tensor hidden, Tensor weight, Tensor labels) -> (Tensor, Tensor)");
  m.impl("fused_ce_fwd", &amd_ops::fused_ce_fwd);

  m.def("soft_ce_fwd(Tensor s, Tensor t) -> (Tensor, Tensor, Tensor)");
  m.impl("soft_ce_fwd", &amd_ops::soft_ce_fwd);
  m.def("soft_ce_bwd(Tensor s, Tensor t, Tensor lse_s, Tensor lse_t, Tensor dloss) -> Tensor");
  m.impl("soft_ce_bwd", &amd_ops::soft_ce_bwd);

  m.def("nf4_dequant(Tensor packed, Tensor absmax, int block_size, int rows, int cols) -> Tensor");
  m.impl("nf4_dequant", &amd_ops::nf4_dequant);
  m.def("fp8_cast(Tensor x, Tensor scale, Tensor(a!) amax_out, bool e5m2) -> Tensor");
  m.impl("fp8_cast", &amd_ops::fp8_cast);
  m.def("fp8_transpose(Tensor x8) -> Tensor");
  m.impl("fp8_transpose", &amd_ops::fp8_transpose);
  m.def("lora_apply(Tensor? y, Tensor x, Tensor A, Tensor B, float scale) -> (Tensor, Tensor)");
  m.impl("lora_apply", &amd_ops::lora_apply);
  m.def("lora_forward(Tensor y, Tensor x, Tensor A, Tensor B, float scale) -> (Tensor, Tensor)");
  m.impl("lora_forward", &amd_ops::lora_forward);
  m.def("lora_linear(Tensor x, Tensor w, Tensor A, Tensor B, float scale) -> (Tensor, Tensor)");
  m.impl("lora_linear", &amd_ops::lora_linear);
  m.def("lora_grads(Tensor g, Tensor x, Tensor A, Tensor B, Tensor tt, float scale) -> (Tensor, Tensor, Tensor, Tensor)");
  m.impl("lora_grads", &amd_ops::lora_grads);
  m.def("linear_dx_extra(Tensor g, Tensor w, Tensor t, Tensor a_t) -> Tensor");
  m.impl("linear_dx_extra", &amd_ops::linear_dx_extra);
  m.def("lora_fused_fwd(Tensor x, Tensor A, Tensor B, float scale) -> Tensor");
  m.impl("lora_fused_fwd", &amd_ops::lora_fused_fwd);
  m.def("sgmv_fused_fwd(Tensor x, Tensor A, Tensor B, Tensor scales, Tensor offs, Tensor tile_map, Tensor? n_tiles=None) -> Tensor");
  m.impl("sgmv_fused_fwd", &amd_ops::sgmv_fused_fwd);

  m.def("build_group_plan(Tensor counts, int M, int bm=128) -> (Tensor, Tensor, Tensor)");
  m.impl("build_group_plan", &amd_ops::build_group_plan);
  m.def("grouped_gemm_nt(Tensor x, Tensor w, Tensor offs, Tensor tile_map, Tensor? n_tiles=None, int bm=128) -> Tensor");
  m.impl("grouped_gemm_nt", &amd_ops::grouped_gemm_nt);
  m.def("grouped_glu(Tensor x, Tensor w, Tensor up, Tensor offs, Tensor tile_map, Tensor? n_tiles=None, int bm=128) -> (Tensor, Tensor, Tensor)");
  m.impl("grouped_glu", &amd_ops::grouped_glu);
  m.def("grouped_gemm_nn(Tensor g, Tensor w, Tensor offs, Tensor tile_map, Tensor? n_tiles=None, int bm=128) -> Tensor");
  m.impl("grouped_gemm_nn", &amd_ops::grouped_gemm_nn);
  m.def("grouped_gemm_cap(int mode, int M, int E, int N, int K) -> int");
  m.impl("grouped_gemm_cap", &amd_ops::grouped_gemm_cap);
  m.def("grouped_gemm_tn(Tensor g, Tensor x, Tensor offs, int E) -> Tensor");
  m.impl("grouped_gemm_tn", &amd_ops::grouped_gemm_tn);
  m.def("small_nt(Tensor x, Tensor w) -> Tensor");
  m.impl("small_nt", &amd_ops::small_nt);
  m.def("small_nn(Tensor g, Tensor w) -> Tensor");
  m.impl("small_nn", &amd_ops::small_nn);
  m.def("small_tn(Tensor g, Tensor x) -> Tensor");
  m.impl("small_tn", &amd_ops::small_tn);
  m.def("small_cut(int rows, int cols, int sum) -> (int, int)", &amd_ops::small_cut);
  m.def("linear_small(Tensor x, Tensor w) -> Tensor", &amd_ops::linear_small);
  m.def("linear_y(Tensor x, Tensor w, bool relu2=False) -> Tensor");
  m.impl("linear_y", &amd_ops::linear_y);
  m.def("linear_glu(Tensor x, Tensor w, Tensor up) -> Tensor");
  m.impl("linear_glu", &amd_ops::linear_glu);
  m.def("linear_y_cut(int T, int N, int K) -> int[]");
  m.impl("linear_y_cut", &amd_ops::linear_y_cut);
  m.def("linear_dw(Tensor g, Tensor x) -> Tensor");
  m.impl("linear_dw", &amd_ops::linear_dw);
  m.def("linear_grad_cut(bool dw, int T, int N, int K) -> int[]");
  m.impl("linear_grad_cut", &amd_ops::linear_grad_cut);
  m.def("linear_dx(Tensor g, Tensor w) -> Tensor");
  m.impl("linear_dx", &amd_ops::linear_dx);
  m.def("grouped_gemm_nt_fp8(Tensor x8, Tensor w8, Tensor offs, Tensor tile_map, Tensor scale, Tensor? n_tiles=None, int bm=128) -> Tensor");
  m.impl("grouped_gemm_nt_fp8", &amd_ops::grouped_gemm_nt_fp8);
  m.def("route_plan(Tensor indices, Tensor probs, int E) -> (Tensor, Tensor, Tensor, Tensor, Tensor)");
  m.impl("route_plan", &amd_ops::route_plan);
  m.def("router_linear(Tensor x, Tensor w) -> Tensor");
  m.impl("router_linear", &amd_ops::router_linear);
  m.def("router_linear_bwd(Tensor d, Tensor x, Tensor w, bool want_dx, bool want_dw) -> (Tensor, Tensor)");
  m.impl("router_linear_bwd", &amd_ops::router_linear_bwd);
  m.def("route_topk(Tensor scores, int K) -> Tensor");
  m.impl("route_topk", &amd_ops::route_topk);
  m.def("route_weights(Tensor scores, Tensor indices, bool norm, float scale, bool bf16_out) -> Tensor");
  m.impl("route_weights", &amd_ops::route_weights);
  m.def("route_weights_bwd(Tensor dprobs, Tensor scores, Tensor indices, bool softmax, bool norm, float scale) -> Tensor");
  m.impl("route_weights_bwd", &amd_ops::route_weights_bwd);
  m.def("expert_load(Tensor indices, int E) -> Tensor");
  m.impl("expert_load", &amd_ops::expert_load);
  m.def("combine_bwd(Tensor g, Tensor y, Tensor src, Tensor order, Tensor probs) -> (Tensor, Tensor)");
  m.impl("combine_bwd", &amd_ops::combine_bwd);
  m.def(
      "grouped_gemm_nn2(Tensor g1, Tensor w1, Tensor g2, Tensor w2, Tensor offs, Tensor tile_map, "
      "Tensor? n_tiles=None, int bm=128) -> Tensor");
  m.impl("grouped_gemm_nn2", &amd_ops::grouped_gemm_nn2);
  m.def("unpermute_combine(Tensor yp, Tensor pos, Tensor probs) -> Tensor");
  m.impl("unpermute_combine", &amd_ops::unpermute_combine);
  m.def("permute_rows(Tensor x, Tensor pos) -> Tensor");
  m.impl("permute_rows", &amd_ops::permute_rows);
  m.def("unpermute_sum(Tensor yp, Tensor pos) -> Tensor");
  m.impl("unpermute_sum", &amd_ops::unpermute_sum);
}
