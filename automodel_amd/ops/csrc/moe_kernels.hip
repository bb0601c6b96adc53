// MoE kernels (CDNA4): fp8 grouped GEMM (MFMA 16x16x32) and fused token permute/unpermute.
// The bf16 grouped GEMM is in grouped_gemm.hip.
//   route_topk / expert_load: the router's choice of experts and how often each was chosen.
//   route_plan: token replicas sorted by expert (stable counting sort), on the device.
//   route_weights: the chosen experts' weights, and the gradient of the router's logits.
//   permute_rows / unpermute_combine: write a token's copies to their places in expert-
//     sorted order, and combine top-k outputs with routing probs, without
//     materializing the repeat_interleave copy; unpermute_sum: the copies' gradient;
//     combine_bwd: the gradients of both factors in one pass.

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <type_traits>

#include "common.h"
#include "ops_api.h"

namespace amd_ops {

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define GG_BM 128
#define GG_BN 128

// LDS tiles: [128 rows][64 cols] bf16, 128-B rows (32 words): rows of equal
// parity share a 32-word bank window; rotating the 16-B slot by (row>>1)&7
// separates the 8 colliding rows of a 16-lane b128 group -> conflict-free.
__device__ __forceinline__ int gg_off(int row, int byte_in_row) {
  return row * 128 + (byte_in_row ^ (((row >> 1) & 7) << 4));
}

static int gg_nfirst() {
  static const int v = []{
    const char* e = getenv("AMD_OPS_GG_NFIRST");
    return e ? atoi(e) : 1;
  }();
  return v;
}

// ---- routing --------------------------------------------------------------
// Stable counting sort of the n = T * K expert choices, in three launches: every wave
// counts its 256 entries per expert, one workgroup turns the [waves, E] counts into first
// places, every wave places its entries in order. Against a radix sort of 64-bit keys, a
// histogram that waits for the host, an inverse permutation and three gathers:
// 65536 choices of 128 experts: 142 us and a wait for the host -> 21 us (29 with the scan's loads one by one; 131072 of
// 512 experts: 142 -> 66); 600 choices: 114 -> 14.
constexpr int ROUTE_CHUNK = 256, ROUTE_MAX_E = 4096;

__device__ __forceinline__ int route_expert(const long* idx, long i, int E) {
  const long e = idx[i];
  return e < 0 ? 0 : e >= E ? E - 1 : (int)e;      // memory stays safe; callers refuse such numbers
}

__global__ __launch_bounds__(64) void route_count_kernel(const long* __restrict__ idx, long n, int E,
                                                         int* __restrict__ count) {
  extern __shared__ int hist[];
  for (int e = threadIdx.x; e < E; e += 64) hist[e] = 0;
  __syncthreads();
  const long i0 = (long)blockIdx.x * ROUTE_CHUNK;
  for (int i = threadIdx.x; i < ROUTE_CHUNK && i0 + i < n; i += 64)
    atomicAdd(&hist[route_expert(idx, i0 + i, E)], 1);
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += 64) count[(long)blockIdx.x * E + e] = hist[e];
}

// count[b][e] -> first place of wave b's entries of expert e; totals per expert
__global__ __launch_bounds__(1024) void route_scan_kernel(int* __restrict__ count, int blocks, int E,
                                                          int* __restrict__ totals) {
  __shared__ int sums[1024], first[ROUTE_MAX_E];
  const int t = threadIdx.x;
  const int cols = min(E, 1024), parts = 1024 / cols;        // experts side by side, strips of blocks
  const int strip = (blocks + parts - 1) / parts;
  for (int e0 = 0; e0 < E; e0 += cols) {                     // strips' sums, then experts' totals
    const int e = e0 + t % cols, part = t / cols;
    int s = 0;
    if (e < E && part < parts)
#pragma unroll 8
      for (int b = part * strip; b < min((part + 1) * strip, blocks); ++b) s += count[(long)b * E + e];
    sums[t] = s;
    __syncthreads();
    if (t < cols && e0 + t < E) {
      int total = 0;
      for (int q = 0; q < parts; ++q) total += sums[q * cols + t];
      totals[e0 + t] = total;
      first[e0 + t] = total;
    }
    __syncthreads();
  }
  // exclusive scan of the totals: a stretch of experts per thread, then over the threads
  const int per = (E + 1023) / 1024;
  int s = 0;
  for (int e = t * per; e < min((t + 1) * per, E); ++e) s += first[e];
  sums[t] = s;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const int v = t >= off ? sums[t - off] : 0;
    __syncthreads();
    sums[t] += v;
    __syncthreads();
  }
  int run = sums[t] - s;
  for (int e = t * per; e < min((t + 1) * per, E); ++e) {
    const int v = first[e];
    first[e] = run;
    run += v;
  }
  __syncthreads();
  for (int e0 = 0; e0 < E; e0 += cols) {
    const int e = e0 + t % cols, part = t / cols;
    const int b0 = part * strip, b1 = min((part + 1) * strip, blocks);
    int sum = 0;
    if (e < E && part < parts)
#pragma unroll 8
      for (int b = b0; b < b1; ++b) sum += count[(long)b * E + e];
    __syncthreads();
    sums[t] = sum;
    __syncthreads();
    if (e < E && part < parts) {
      int place = first[e];
      for (int q = 0; q < part; ++q) place += sums[q * cols + t % cols];
      for (int b = b0; b < b1; b += 8) {                     // (one by one each load waited for the last store)
        int c[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) c[j] = b + j < b1 ? count[(long)(b + j) * E + e] : 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (b + j < b1) count[(long)(b + j) * E + e] = place;
          place += c[j];
        }
      }
    }
  }
}

__global__ __launch_bounds__(64) void route_place_kernel(const long* __restrict__ idx,
                                                         const float* __restrict__ probs, long n, int E,
                                                         int K, const int* __restrict__ first,
                                                         int* __restrict__ order, int* __restrict__ src,
                                                         int* __restrict__ pos,
                                                         float* __restrict__ perm_probs) {
  extern __shared__ int next[];
  for (int e = threadIdx.x; e < E; e += 64) next[e] = first[(long)blockIdx.x * E + e];
  __syncthreads();
  const int bits = 32 - __clz(E);
  for (int c = 0; c < ROUTE_CHUNK; c += 64) {
    const long i = (long)blockIdx.x * ROUTE_CHUNK + c + threadIdx.x;
    const bool in = i < n;
    const int e = in ? route_expert(idx, i, E) : E;
    unsigned long long same = ~0ull;                         // lanes with the same expert
    for (int b = 0; b < bits; ++b) {
      const unsigned long long m = __ballot((e >> b) & 1);
      same &= (e >> b) & 1 ? m : ~m;
    }
    const unsigned long long below = same & ((1ull << threadIdx.x) - 1);
    int at = 0;
    if (in) at = next[e] + __popcll(below);
    __syncthreads();
    if (in && below == 0) next[e] += __popcll(same);
    __syncthreads();
    if (in) {
      order[at] = (int)i;
      src[at] = (int)(i / K);
      pos[i] = at;
      perm_probs[at] = probs[i];
    }
  }
}

// ---- the router's choice ---------------------------------------------------
// The K largest of E scores of each token, a wave per token: a lane holds V neighbouring
// scores as unsigned keys in the order of the floats (NaN above all, as torch.topk has it);
// K times, the wave's largest key is taken out, the lowest expert first where scores are equal.
// One read of the scores and a chain of K reductions; torch.topk selects by radix, a
// workgroup per row, and sorts in a second launch.
// 8192 x 128, K 8: 63 -> 7.4 us; 3003 x 64, K 6: 25 -> 4.6; 1 x 64: 14 -> 4.7. The chain grows
// with K and V, and the lead shrinks: 4096 x 512, K 8: 95 -> 8.8; 16384 x 512, K 32:
// 235 -> 55; nothing larger was measured, and larger ones stay with torch.topk.
constexpr int CHOICE_MAX_E = 512, CHOICE_MAX_K = 32;

template <int V>
__global__ __launch_bounds__(256) void route_topk_kernel(const float* __restrict__ scores, int T, int E,
                                                         int K, long* __restrict__ out) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= T) return;
  unsigned key[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int e = lane * V + j;
    key[j] = 0;                                  // below every score, -inf too
    if (e < E) {
      const float s = scores[(long)t * E + e];
      const unsigned u = __float_as_uint(s);
      key[j] = s == s ? u ^ (u >> 31 ? ~0u : 1u << 31) : ~0u;
    }
  }
  int mine = 0;
  for (int k = 0; k < K; ++k) {
    unsigned top = key[0];
#pragma unroll
    for (int j = 1; j < V; ++j) top = max(top, key[j]);
    unsigned m = top;
#pragma unroll
    for (int o = 32; o; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o, 64));
    const int owner = __ffsll((unsigned long long)__ballot(top == m)) - 1;
    int at = 0;
#pragma unroll
    for (int j = V - 1; j >= 0; --j) at = key[j] == m ? j : at;
#pragma unroll
    for (int j = 0; j < V; ++j)
      if (lane == owner && j == at) key[j] = 0;
    const int e = owner * V + __shfl(at, owner, 64);
    if (lane == k) mine = e;
  }
  if (lane < K) out[(long)t * K + lane] = mine;
}

// scores [T, E] -> experts [T, K], the largest score first
at::Tensor route_topk(const at::Tensor& scores, int64_t K) {
  TORCH_CHECK(scores.is_cuda() && scores.dim() == 2 && scores.scalar_type() == at::kFloat &&
                  scores.is_contiguous(), "route_topk: scores [T,E] float32");
  const long T = scores.size(0), E = scores.size(1);
  TORCH_CHECK(E <= CHOICE_MAX_E && K >= 1 && K <= std::min<long>(E, CHOICE_MAX_K), "route_topk: 1 to ",
              CHOICE_MAX_K, " of at most ", CHOICE_MAX_E, " experts");
  TORCH_CHECK(T < (1l << 31) - 4, "route_topk: too many tokens");
  const c10::DeviceGuard guard(scores.device());
  auto out = at::empty({T, K}, scores.options().dtype(at::kLong));
  if (!T) return out;
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)((T + 3) / 4)), dim3(256), 0, stream, scores.data_ptr<float>(),
                       (int)T, (int)E, (int)K, out.data_ptr<long>());
  };
  if (E <= 64) launch(route_topk_kernel<1>);
  else if (E <= 128) launch(route_topk_kernel<2>);
  else if (E <= 256) launch(route_topk_kernel<4>);
  else launch(route_topk_kernel<8>);
  HIP_CHECK_KERNEL();
  return out;
}

// ---- the chosen experts' weights ---------------------------------------------
// probs[t, k] = scores[t, idx[t, k]], over their sum if NORM (1e-20 at least), times scale; and the gradient of
// the router's logits, whose softmax or sigmoid the scores are. A wave per token. What these are bound by is launches:
// torch's are 6 of 5 us forward and 16 backward (8192 x 128, K 8: 31 -> 2.7 us, and 79 -> 4.9).
template <bool NORM, typename Out>
__global__ __launch_bounds__(256) void route_weights_kernel(const float* __restrict__ scores,
                                                            const long* __restrict__ idx, int T, int E, int K,
                                                            float scale, Out* __restrict__ probs) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= T) return;
  const float s = lane < K ? scores[(long)t * E + route_expert(idx, (long)t * K + lane, E)] : 0.f;
  float p = s;
  if constexpr (NORM) {
    const float sum = wave_reduce_sum(s);
    p = s / (sum < 1e-20f ? 1e-20f : sum);                  // (a NaN stays one)
  }
  if (lane >= K) return;
  if constexpr (std::is_same_v<Out, float>) probs[(long)t * K + lane] = p * scale;
  else probs[(long)t * K + lane] = f2bf(p * scale);
}

template <bool NORM, bool SOFTMAX, typename In>
__global__ __launch_bounds__(256) void route_weights_bwd_kernel(const In* __restrict__ dprobs,
                                                                const float* __restrict__ scores,
                                                                const long* __restrict__ idx, int T, int E, int K,
                                                                float scale, float* __restrict__ dlogits) {
  __shared__ float rows[4][CHOICE_MAX_E];
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= T) return;                                       // (waves do not meet)
  float* ds = rows[threadIdx.x >> 6];
  for (int e = lane; e < E; e += 64) ds[e] = 0.f;
  float s = 0.f, d = 0.f;
  int e = 0;
  if (lane < K) {
    e = route_expert(idx, (long)t * K + lane, E);
    s = scores[(long)t * E + e];
    if constexpr (std::is_same_v<In, float>) d = dprobs[(long)t * K + lane] * scale;
    else d = bf2f(dprobs[(long)t * K + lane]) * scale;
  }
  if constexpr (NORM) {
    const float sum = wave_reduce_sum(s), dot = wave_reduce_sum(lane < K ? d * s : 0.f);
    const float n = sum < 1e-20f ? 1e-20f : sum;
    d = d / n - (sum >= 1e-20f ? dot / (n * n) : 0.f);
  }
  float all = 0.f;
  if constexpr (SOFTMAX) all = wave_reduce_sum(lane < K ? d * s : 0.f);
  __builtin_amdgcn_wave_barrier();
  if (lane < K) atomicAdd(&ds[e], d);                       // (one expert, one lane: sums in no order only of doubled ones)
  __builtin_amdgcn_wave_barrier();
  for (int c = lane; c < E; c += 64) {
    const float y = scores[(long)t * E + c], g = ds[c];
    dlogits[(long)t * E + c] = SOFTMAX ? (g - all) * y : g * (1.f - y) * y;
  }
}

static void check_weights(const char* name, const at::Tensor& scores, const at::Tensor& idx) {
  TORCH_CHECK(scores.is_cuda() && scores.dim() == 2 && scores.scalar_type() == at::kFloat && scores.is_contiguous() &&
                  idx.device() == scores.device() && idx.dim() == 2 && idx.scalar_type() == at::kLong &&
                  idx.is_contiguous() && idx.size(0) == scores.size(0), name, ": scores [T,E] float32, indices [T,K]");
  TORCH_CHECK(scores.size(1) >= 1 && scores.size(1) <= CHOICE_MAX_E && idx.size(1) >= 1 && idx.size(1) <= CHOICE_MAX_K &&
                  scores.size(0) < (1l << 31) - 4, name, ": at most ", CHOICE_MAX_K, " of ", CHOICE_MAX_E, " experts");
}

at::Tensor route_weights(const at::Tensor& scores, const at::Tensor& idx, bool norm, double scale, bool bf16_out) {
  check_weights("route_weights", scores, idx);
  const c10::DeviceGuard guard(scores.device());
  auto probs = at::empty(idx.sizes(), scores.options().dtype(bf16_out ? at::kBFloat16 : at::kFloat));
  const int T = (int)scores.size(0);
  if (!T) return probs;
  auto launch = [&](auto norm_, auto* out) {
    hipLaunchKernelGGL((route_weights_kernel<decltype(norm_)::value, std::remove_reference_t<decltype(*out)>>),
                       dim3((T + 3) / 4), dim3(256), 0, c10::hip::getCurrentHIPStream().stream(),
                       scores.data_ptr<float>(), idx.data_ptr<long>(), T, (int)scores.size(1), (int)idx.size(1),
                       (float)scale, out);
  };
  auto typed = [&](auto* out) { norm ? launch(std::true_type{}, out) : launch(std::false_type{}, out); };
  if (bf16_out) typed(reinterpret_cast<bf16*>(probs.data_ptr()));
  else typed(probs.data_ptr<float>());
  HIP_CHECK_KERNEL();
  return probs;
}

at::Tensor route_weights_bwd(const at::Tensor& dprobs, const at::Tensor& scores, const at::Tensor& idx, bool softmax,
                             bool norm, double scale) {
  check_weights("route_weights_bwd", scores, idx);
  TORCH_CHECK(dprobs.device() == scores.device() && dprobs.sizes() == idx.sizes() && dprobs.is_contiguous() &&
                  (dprobs.scalar_type() == at::kFloat || dprobs.scalar_type() == at::kBFloat16),
              "route_weights_bwd: dprobs [T,K] bf16 or float32");
  const c10::DeviceGuard guard(scores.device());
  auto dlogits = at::empty_like(scores);
  const int T = (int)scores.size(0);
  if (!T) return dlogits;
  auto launch = [&](auto norm_, auto softmax_, const auto* in) {
    hipLaunchKernelGGL((route_weights_bwd_kernel<decltype(norm_)::value, decltype(softmax_)::value,
                                                 std::remove_cv_t<std::remove_reference_t<decltype(*in)>>>),
                       dim3((T + 3) / 4), dim3(256), 0, c10::hip::getCurrentHIPStream().stream(), in,
                       scores.data_ptr<float>(), idx.data_ptr<long>(), T, (int)scores.size(1), (int)idx.size(1),
                       (float)scale, dlogits.data_ptr<float>());
  };
  auto typed = [&](const auto* in) {
    using Yes = std::true_type;
    using No = std::false_type;
    if (norm) softmax ? launch(Yes{}, Yes{}, in) : launch(Yes{}, No{}, in);
    else softmax ? launch(No{}, Yes{}, in) : launch(No{}, No{}, in);
  };
  if (dprobs.scalar_type() == at::kBFloat16) typed(reinterpret_cast<const bf16*>(dprobs.data_ptr()));
  else typed(dprobs.data_ptr<float>());
  HIP_CHECK_KERNEL();
  return dlogits;
}

// How often each expert was chosen, as float. Every workgroup counts 4096 choices in LDS and adds
// its counts (whole numbers: exact in any order); adding every choice to its place in memory
// queues n / E additions there. 65536 choices of 128: 45 -> 8.2 us
// with the fill of the result, 524288 of 512: 190 -> 8.2.
constexpr int LOAD_CHUNK = 4096;

__global__ __launch_bounds__(256) void expert_load_kernel(const long* __restrict__ idx, long n, int E,
                                                          float* __restrict__ load) {
  extern __shared__ int hist[];
  for (int e = threadIdx.x; e < E; e += 256) hist[e] = 0;
  __syncthreads();
  const long end = min(n, ((long)blockIdx.x + 1) * LOAD_CHUNK);
  for (long i = (long)blockIdx.x * LOAD_CHUNK + threadIdx.x; i < end; i += 256)
    atomicAdd(&hist[route_expert(idx, i, E)], 1);
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += 256)
    if (hist[e]) atomicAdd(&load[e], (float)hist[e]);
}

at::Tensor expert_load(const at::Tensor& indices, int64_t E) {
  TORCH_CHECK(indices.is_cuda() && indices.scalar_type() == at::kLong && indices.is_contiguous(),
              "expert_load: indices int64");
  TORCH_CHECK(E >= 1 && E <= ROUTE_MAX_E, "expert_load: 1 to ", ROUTE_MAX_E, " experts");
  const long n = indices.numel();
  TORCH_CHECK(n < (1l << 31), "expert_load: too many choices");
  const c10::DeviceGuard guard(indices.device());
  auto load = at::zeros({E}, indices.options().dtype(at::kFloat));
  if (n)
    hipLaunchKernelGGL(expert_load_kernel, dim3((unsigned)((n + LOAD_CHUNK - 1) / LOAD_CHUNK)), dim3(256),
                       E * sizeof(int), c10::hip::getCurrentHIPStream().stream(), indices.data_ptr<long>(),
                       n, (int)E, load.data_ptr<float>());
  HIP_CHECK_KERNEL();
  return load;
}

// indices [T, K] of experts, probs [T, K] -> counts [E]; per place in expert order: the
// flat choice, its token, its prob; and each choice's place [T, K]
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor> route_plan(
    const at::Tensor& indices, const at::Tensor& probs, int64_t E) {
  TORCH_CHECK(indices.is_cuda() && indices.dim() == 2 && indices.scalar_type() == at::kLong &&
                  indices.is_contiguous(), "route_plan: indices [T,K] int64");
  TORCH_CHECK(probs.sizes() == indices.sizes() && probs.scalar_type() == at::kFloat && probs.is_contiguous(),
              "route_plan: probs [T,K] float32");
  TORCH_CHECK(E >= 1 && E <= ROUTE_MAX_E, "route_plan: 1 to ", ROUTE_MAX_E, " experts");
  const long n = indices.numel();
  TORCH_CHECK(n < (1l << 31), "route_plan: too many choices");
  auto ints = indices.options().dtype(at::kInt);
  auto counts = at::empty({E}, ints), order = at::empty({n}, ints), src = at::empty({n}, ints),
       pos = at::empty(indices.sizes(), ints);
  auto perm_probs = at::empty({n}, probs.options());
  const int blocks = (int)((n + ROUTE_CHUNK - 1) / ROUTE_CHUNK);
  auto work = at::empty({std::max(blocks, 1), E}, ints);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const long* idx = indices.data_ptr<long>();
  if (blocks)
    hipLaunchKernelGGL(route_count_kernel, dim3(blocks), dim3(64), E * sizeof(int), stream, idx, n, (int)E,
                       work.data_ptr<int>());
  hipLaunchKernelGGL(route_scan_kernel, dim3(1), dim3(1024), 0, stream, work.data_ptr<int>(), blocks, (int)E,
                     counts.data_ptr<int>());
  if (blocks)
    hipLaunchKernelGGL(route_place_kernel, dim3(blocks), dim3(64), E * sizeof(int), stream, idx,
                       probs.data_ptr<float>(), n, (int)E, (int)indices.size(1), work.data_ptr<int>(),
                       order.data_ptr<int>(), src.data_ptr<int>(), pos.data_ptr<int>(),
                       perm_probs.data_ptr<float>());
  HIP_CHECK_KERNEL();
  return {counts, order, src, pos, perm_probs};
}

// backward of the combine: dy[i] = g[src[i]] * p[i], dprobs[order[i]] = sum(g[src[i]] * y[i]);
// a wave per place, one pass over y. Bound by reading y and g and writing dy (65536 x 2048: 115 us,
// 805 MB; a gather and eight passes of torch operations took 830 us).
__global__ __launch_bounds__(256) void combine_bwd_kernel(const bf16* __restrict__ g,
                                                          const bf16* __restrict__ y,
                                                          const int* __restrict__ src,
                                                          const int* __restrict__ order,
                                                          const float* __restrict__ p,
                                                          bf16* __restrict__ dy, float* __restrict__ dp,
                                                          int H, long M) {
  const long i = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= M) return;
  const int lane = threadIdx.x & 63;
  const bf16* gr = g + (long)src[i] * H;
  const float w = p[i];
  float s = 0.f;
#pragma unroll 4
  for (int c = lane * 8; c < H; c += 512) {
    const bf16x8 gv = *reinterpret_cast<const bf16x8*>(gr + c);
    const bf16x8 yv = *reinterpret_cast<const bf16x8*>(y + i * H + c);
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float gf = bf2f(gv.v[j]);
      s = fmaf(gf, bf2f(yv.v[j]), s);
      o.v[j] = f2bf(gf * w);
    }
    *reinterpret_cast<bf16x8*>(dy + i * H + c) = o;
  }
  s = wave_reduce_sum(s);
  if (lane == 0) dp[order[i]] = s;
}

std::tuple<at::Tensor, at::Tensor> combine_bwd(const at::Tensor& g, const at::Tensor& y,
                                               const at::Tensor& src, const at::Tensor& order,
                                               const at::Tensor& probs) {
  const long M = y.size(0);
  const int H = y.size(1);
  TORCH_CHECK(g.is_cuda() && g.dim() == 2 && g.size(1) == H && H % 8 == 0 && g.is_contiguous() &&
                  y.is_contiguous() && g.scalar_type() == at::kBFloat16 && y.scalar_type() == at::kBFloat16,
              "combine_bwd: g [T,H], y [M,H] bf16, H%8==0");
  TORCH_CHECK(src.numel() == M && order.numel() == M && probs.numel() == M &&
                  src.scalar_type() == at::kInt && order.scalar_type() == at::kInt &&
                  probs.scalar_type() == at::kFloat, "combine_bwd: one place per row of y");
  auto dy = at::empty_like(y);
  auto dp = at::empty({M}, probs.options());
  if (M == 0) return {dy, dp};
  hipLaunchKernelGGL(combine_bwd_kernel, dim3((unsigned)((M + 3) / 4)), dim3(256), 0,
                     c10::hip::getCurrentHIPStream().stream(),
                     reinterpret_cast<const bf16*>(g.data_ptr()),
                     reinterpret_cast<const bf16*>(y.data_ptr()), src.data_ptr<int>(),
                     order.data_ptr<int>(), probs.data_ptr<float>(),
                     reinterpret_cast<bf16*>(dy.data_ptr()), dp.data_ptr<float>(), H, M);
  HIP_CHECK_KERNEL();
  return {dy, dp};
}

// ---- fused permute / unpermute -------------------------------------------
// A token's choices in groups of 8, of which the last has TAIL (1 to 8): f(first of the group, constant of its size).
// The loads or stores of a group are expanded and go out together, whatever the number of choices.
template <int TAIL, typename F>
__device__ __forceinline__ void choice_groups(int topk, F&& f) {
  int k = 0;
  for (; k + TAIL < topk; k += 8) f(k, std::integral_constant<int, 8>{});
  f(k, std::integral_constant<int, TAIL>{});
}

// y[pos[t, k]] = x[t] for all k: a token's row is read once and its copies' stores go out together, instead of a
// workgroup for each copy (65536 rows of 2048 columns, 8 a token: 74 us, now 47; one by one 5 and 9 a token were 69 and 58,
// now 60 and 48)
template <int TAIL>
__global__ void permute_rows_kernel(const bf16* __restrict__ x, bf16* __restrict__ y, const int* __restrict__ pos, int H,
                                    int topk) {
  const long t = blockIdx.x;
  const int* at = pos + t * topk;
  for (int c = threadIdx.x * 8; c < H; c += blockDim.x * 8) {
    const bf16x8 v = *reinterpret_cast<const bf16x8*>(x + t * H + c);
    choice_groups<TAIL>(topk, [&](int k0, auto n) __attribute__((always_inline)) {
#pragma unroll
      for (int k = 0; k < decltype(n)::value; ++k) *reinterpret_cast<bf16x8*>(y + (long)at[k0 + k] * H + c) = v;
    });
  }
}

// combine: out[t, :] = sum_k probs[t, k] * yp[pos[t*K + k], :], or without probs the sum alone
template <int TAIL>
__global__ void unpermute_combine_kernel(const bf16* __restrict__ yp,
                                         bf16* __restrict__ out,
                                         const int* __restrict__ pos,
                                         const float* __restrict__ probs,
                                         int H, int topk, long T) {
  const long t = blockIdx.x;
  bf16* orow = out + t * (long)H;
  for (int c = threadIdx.x * 8; c < H; c += blockDim.x * 8) {
    float accv[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    choice_groups<TAIL>(topk, [&](int k0, auto n) __attribute__((always_inline)) {
      constexpr int N = decltype(n)::value;
      const long at = t * topk + k0;
      bf16x8 v[N];
#pragma unroll
      for (int k = 0; k < N; ++k) v[k] = *reinterpret_cast<const bf16x8*>(yp + (long)pos[at + k] * H + c);
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const float p = probs ? probs[at + k] : 1.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) accv[j] += p * bf2f(v[k].v[j]);
      }
    });
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o.v[j] = f2bf(accv[j]);
    *reinterpret_cast<bf16x8*>(orow + c) = o;
  }
}

// f(constant of the last group's size)
template <typename F>
static void with_tail(int topk, F&& f) {
  switch ((topk - 1) % 8) {
    case 0: return f(std::integral_constant<int, 1>{});
    case 1: return f(std::integral_constant<int, 2>{});
    case 2: return f(std::integral_constant<int, 3>{});
    case 3: return f(std::integral_constant<int, 4>{});
    case 4: return f(std::integral_constant<int, 5>{});
    case 5: return f(std::integral_constant<int, 6>{});
    case 6: return f(std::integral_constant<int, 7>{});
    default: return f(std::integral_constant<int, 8>{});
  }
}

// x [T, H], pos [T, K]: the place of each token's copies, every place once -> [T * K, H]
at::Tensor permute_rows(const at::Tensor& x, const at::Tensor& pos) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.scalar_type() == at::kBFloat16 && x.is_contiguous() && x.size(1) % 8 == 0 &&
                  pos.device() == x.device() && pos.dim() == 2 && pos.is_contiguous() && pos.scalar_type() == at::kInt &&
                  pos.size(0) == x.size(0), "permute_rows: x bf16 [T, H], H%8==0, pos int32 [T, K]");
  const long T = x.size(0);
  const int H = x.size(1), topk = pos.size(1);
  auto y = at::empty({T * topk, (long)H}, x.options());
  if (y.numel() == 0) return y;
  with_tail(topk, [&](auto tail) {
    hipLaunchKernelGGL((permute_rows_kernel<decltype(tail)::value>), dim3(T), dim3(std::min(256, H / 8)), 0,
                       c10::hip::getCurrentHIPStream().stream(), reinterpret_cast<const bf16*>(x.data_ptr()),
                       reinterpret_cast<bf16*>(y.data_ptr()), pos.data_ptr<int>(), H, topk);
  });
  HIP_CHECK_KERNEL();
  return y;
}

static at::Tensor combine(const at::Tensor& yp, const int* pos, const float* probs, long T, int topk) {
  const int H = yp.size(1);
  auto out = at::empty({T, (long)H}, yp.options());
  if (T == 0) return out;
  if (topk == 0) return out.zero_();
  with_tail(topk, [&](auto tail) {
    hipLaunchKernelGGL((unpermute_combine_kernel<decltype(tail)::value>), dim3(T), dim3(std::min(256, H / 8)), 0,
                       c10::hip::getCurrentHIPStream().stream(), reinterpret_cast<const bf16*>(yp.data_ptr()),
                       reinterpret_cast<bf16*>(out.data_ptr()), pos, probs, H, topk, T);
  });
  HIP_CHECK_KERNEL();
  return out;
}

at::Tensor unpermute_combine(const at::Tensor& yp, const at::Tensor& pos,
                             const at::Tensor& probs) {
  return combine(yp, pos.data_ptr<int>(), probs.data_ptr<float>(), probs.size(0), (int)probs.size(1));
}

// rows yp [T * K, H] in expert order -> the sum of each token's, pos [T, K]
at::Tensor unpermute_sum(const at::Tensor& yp, const at::Tensor& pos) {
  TORCH_CHECK(yp.is_cuda() && yp.dim() == 2 && yp.scalar_type() == at::kBFloat16 && yp.is_contiguous() &&
                  yp.size(1) % 8 == 0 && pos.device() == yp.device() && pos.dim() == 2 && pos.is_contiguous() &&
                  pos.scalar_type() == at::kInt, "unpermute_sum: yp bf16 [n, H], H%8==0, pos int32 [T, K]");
  return combine(yp, pos.data_ptr<int>(), nullptr, pos.size(0), (int)pos.size(1));
}

// ===========================================================================
// fp8 grouped GEMM forward (SURVEY §2.5 last gap: the reference's MXFP8
// grouped path, moe/fp8_utils.py). Tensorwise-scaled OCP e4m3 operands,
// __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8 (bf16 MFMA rate, HALF the
// HBM/LDS bytes — the bf16 grouped kernels are memory-wait-bound per
// profiles/gg_r2_pmc_counters.csv, so fp8 wins on bandwidth, not rate).
// BK = 128 fp8 bytes per stage: rows are 128 B exactly like the bf16
// tiles, so the proven gg_off swizzle carries over unchanged.
// ===========================================================================

typedef long fp8x8;   // 8 packed e4m3 bytes = one MFMA operand

__global__ __launch_bounds__(256) void grouped_gemm_nt_fp8_kernel(
    const unsigned char* __restrict__ x, const unsigned char* __restrict__ w,
    bf16* __restrict__ y, const int* __restrict__ tile_map,
    const int* __restrict__ offs, const int* __restrict__ n_tiles,
    int K, int N, const float* __restrict__ scale_p, int nfirst) {
  const int tb = nfirst ? (int)blockIdx.y : (int)blockIdx.x;
  const int nb = nfirst ? (int)blockIdx.x : (int)blockIdx.y;
  if (n_tiles != nullptr && tb >= n_tiles[0]) return;
  const float scale = scale_p[0];
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* xa = smem;                  // [128 m][128 k-bytes] 16 KiB
  char* wb = smem + GG_BM * 128;

  const int e = tile_map[2 * tb];
  const int m0 = tile_map[2 * tb + 1];
  const int m_end = offs[e + 1];
  const int n0 = nb * GG_BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = tid >> 6;
  const int l16 = lane & 15;
  const int kq = lane >> 4;

  const long wbase = (long)e * N * K;

  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

  const int row0 = tid / 8;          // 8 x 16-B chunks per 128-B row
  const int c0 = (tid % 8) * 16;

  for (int k0 = 0; k0 < K; k0 += 128) {
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      const int row = row0 + rr * 32;
      const int m = m0 + row;
      int4 xv;
      if (m < m_end) {
        xv = *reinterpret_cast<const int4*>(x + (long)m * K + k0 + c0);
      } else {
        xv = make_int4(0, 0, 0, 0);
      }
      *reinterpret_cast<int4*>(xa + gg_off(row, c0)) = xv;
      int4 wv = *reinterpret_cast<const int4*>(
          w + wbase + (long)(n0 + row) * K + k0 + c0);
      *reinterpret_cast<int4*>(wb + gg_off(row, c0)) = wv;
    }
    __syncthreads();

#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      fp8x8 a[4], b[4];
      const int arow = (wid >> 1) * 64;
      const int brow = (wid & 1) * 64;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = *reinterpret_cast<const fp8x8*>(
            xa + gg_off(arow + i * 16 + l16, kk * 32 + kq * 8));
        b[i] = *reinterpret_cast<const fp8x8*>(
            wb + gg_off(brow + i * 16 + l16, kk * 32 + kq * 8));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
              a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }

  const int mw = m0 + (wid >> 1) * 64;
  const int nw = n0 + (wid & 1) * 64;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = mw + i * 16 + kq * 4 + r;
      if (m < m_end) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          y[(long)m * N + nw + j * 16 + l16] = f2bf(acc[i][j][r] * scale);
      }
    }
  }
}

// 256x256 fp8 big-tile (8 waves, 64 KiB LDS): the production MoE tile.
__global__ __launch_bounds__(512, 1) void grouped_gemm_nt_fp8_big_kernel(
    const unsigned char* __restrict__ x, const unsigned char* __restrict__ w,
    bf16* __restrict__ y, const int* __restrict__ tile_map,
    const int* __restrict__ offs, const int* __restrict__ n_tiles,
    int K, int N, const float* __restrict__ scale_p, int nfirst) {
  const int tb = nfirst ? (int)blockIdx.y : (int)blockIdx.x;
  const int nb = nfirst ? (int)blockIdx.x : (int)blockIdx.y;
  if (n_tiles != nullptr && tb >= n_tiles[0]) return;
  const float scale = scale_p[0];
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* xa = smem;                    // [256 m][128 k-bytes] 32 KiB
  char* wb = smem + 256 * 128;

  const int e = tile_map[2 * tb];
  const int m0 = tile_map[2 * tb + 1];
  const int m_end = offs[e + 1];
  const int n0 = nb * 256;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = tid >> 6;
  const int l16 = lane & 15;
  const int kq = lane >> 4;

  const long wbase = (long)e * N * K;

  f32x4 acc[4][8];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

  const int row0 = tid / 8;            // 64 rows per pass (of 256)
  const int c0 = (tid % 8) * 16;

  for (int k0 = 0; k0 < K; k0 += 128) {
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      const int row = row0 + rr * 64;
      const int m = m0 + row;
      int4 xv;
      if (m < m_end) {
        xv = *reinterpret_cast<const int4*>(x + (long)m * K + k0 + c0);
      } else {
        xv = make_int4(0, 0, 0, 0);
      }
      *reinterpret_cast<int4*>(xa + gg_off(row, c0)) = xv;
      int4 wv = *reinterpret_cast<const int4*>(
          w + wbase + (long)(n0 + row) * K + k0 + c0);
      *reinterpret_cast<int4*>(wb + gg_off(row, c0)) = wv;
    }
    __syncthreads();

#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      fp8x8 a[4], b[8];
      const int arow = (wid >> 1) * 64;
      const int brow = (wid & 1) * 128;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        a[i] = *reinterpret_cast<const fp8x8*>(
            xa + gg_off(arow + i * 16 + l16, kk * 32 + kq * 8));
#pragma unroll
      for (int j = 0; j < 8; ++j)
        b[j] = *reinterpret_cast<const fp8x8*>(
            wb + gg_off(brow + j * 16 + l16, kk * 32 + kq * 8));
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(
              a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }

  const int mw = m0 + (wid >> 1) * 64;
  const int nw = n0 + (wid & 1) * 128;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = mw + i * 16 + kq * 4 + r;
      if (m < m_end) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          y[(long)m * N + nw + j * 16 + l16] = f2bf(acc[i][j][r] * scale);
      }
    }
  }
}

at::Tensor grouped_gemm_nt_fp8(const at::Tensor& x8, const at::Tensor& w8,
                               const at::Tensor& offs, const at::Tensor& tile_map,
                               const at::Tensor& scale,
                               const std::optional<at::Tensor>& n_tiles,
                               int64_t bm) {
  TORCH_CHECK(scale.is_cuda() && scale.scalar_type() == at::kFloat && scale.numel() == 1,
              "scale: 1-elem float32 device tensor (combined sx*sw dequant)");
  TORCH_CHECK(x8.is_cuda() && x8.dim() == 2 && x8.element_size() == 1,
              "grouped_gemm_nt_fp8: x8 [M,K] e4m3 bytes");
  TORCH_CHECK(w8.dim() == 3 && w8.element_size() == 1, "w8 [E,N,K] e4m3 bytes");
  const long M = x8.size(0);
  const int K = x8.size(1), N = w8.size(1);
  TORCH_CHECK(K == w8.size(2), "K mismatch");
  TORCH_CHECK(K % 128 == 0 && N % GG_BN == 0, "need K%128==0, N%128==0");
  auto y = at::empty({M, (long)N},
                     x8.options().dtype(at::kBFloat16));
  const int n_mtiles = tile_map.size(0);
  if (n_mtiles == 0 || M == 0) return y;
  auto stream = c10::hip::getCurrentHIPStream();
  const int* ntp = n_tiles.has_value() ? n_tiles->data_ptr<int>() : nullptr;
  if (bm == 256) {
    TORCH_CHECK(N % 256 == 0, "big-tile fp8 nt needs N%256==0");
    const int nfirstb = gg_nfirst();
    const dim3 gridb = nfirstb ? dim3(N / 256, n_mtiles) : dim3(n_mtiles, N / 256);
    hipLaunchKernelGGL(grouped_gemm_nt_fp8_big_kernel, gridb, dim3(512),
                       2 * 256 * 128, stream.stream(),
                       reinterpret_cast<const unsigned char*>(x8.data_ptr()),
                       reinterpret_cast<const unsigned char*>(w8.data_ptr()),
                       reinterpret_cast<bf16*>(y.data_ptr()),
                       tile_map.data_ptr<int>(), offs.data_ptr<int>(), ntp, K, N,
                       scale.data_ptr<float>(), nfirstb);
    HIP_CHECK_KERNEL();
    return y;
  }
  const int nfirst = gg_nfirst();
  const dim3 grid = nfirst ? dim3(N / GG_BN, n_mtiles) : dim3(n_mtiles, N / GG_BN);
  hipLaunchKernelGGL(grouped_gemm_nt_fp8_kernel, grid, dim3(256),
                     2 * GG_BM * 128, stream.stream(),
                     reinterpret_cast<const unsigned char*>(x8.data_ptr()),
                       reinterpret_cast<const unsigned char*>(w8.data_ptr()),
                     reinterpret_cast<bf16*>(y.data_ptr()),
                     tile_map.data_ptr<int>(), offs.data_ptr<int>(), ntp, K, N,
                     scale.data_ptr<float>(), nfirst);
  HIP_CHECK_KERNEL();
  return y;
}

}  // namespace amd_ops
