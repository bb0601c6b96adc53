// Fused AdamW step (CDNA4): bf16 params + fp32 master weights + fp32 moments.
// Semantics match torch.optim.AdamW exactly (decoupled weight decay applied
// multiplicatively before the moment update) so the optimizer parity test can
// compare against torch. Replaces the reference's Apex FusedAdam path
// (nemo_automodel/components/optim/optimizer.py:297).
//
// Memory-bound: 14 B read + 14 B written per element in bf16 with f32 states; float4 /
// bf16x4 vectors, several in flight.

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include "common.h"
#include "ops_api.h"

namespace amd_ops {

// All bf16 parameters with f32 states of a group, as many per launch as fit its arguments;
// a workgroup takes a chunk of one of them, all its loads in flight at once. One launch per
// parameter, each with a loop over 4096 workgroups, left the step of a small model to the
// launches (10.5 million elements in 20 tensors: 122 us, now 46) and read and wrote large
// ones slower (134 million: 902 us, 4.2 TB/s; now 671, 5.6; chunks of 4 and 16 times the
// size 718 and 735).
//
// STREAM: states that the last-level cache (256 MB) does not hold until the next step leave
// no trace in it (707 us without, of the 671); smaller ones stay (54 us with, of the 46).
constexpr int ADAMW_TENSORS = 40;
constexpr int ADAMW_UNROLL = 4, ADAMW_CHUNK = 256 * 4 * ADAMW_UNROLL;
constexpr long ADAMW_CACHED = (256l << 20) / 12;        // elements with 12 bytes of state

struct AdamwTensors {
  bf16* p[ADAMW_TENSORS];
  const bf16* g[ADAMW_TENSORS];
  float* master[ADAMW_TENSORS];
  float* m[ADAMW_TENSORS];
  float* v[ADAMW_TENSORS];
  unsigned first[ADAMW_TENSORS];        // workgroup that a tensor begins with
  long n[ADAMW_TENSORS];                // a multiple of 4
  float inv_bc1[ADAMW_TENSORS], inv_sqrt_bc2[ADAMW_TENSORS];
  int count;
};

typedef float adamw_f32x4 __attribute__((ext_vector_type(4)));

template <bool STREAM>
__global__ __launch_bounds__(256) void adamw_bf16_kernel(const AdamwTensors a, float lr, float b1,
                                                         float b2, float eps, float wd_factor) {
  int t = 0;
  while (t + 1 < a.count && blockIdx.x >= a.first[t + 1]) ++t;
  const long n = a.n[t];
  const long i0 = (long)(blockIdx.x - a.first[t]) * ADAMW_CHUNK;
  const long end = min(i0 + ADAMW_CHUNK, n);
  bf16* __restrict__ p = a.p[t];
  const bf16* __restrict__ g = a.g[t];
  float *__restrict__ master = a.master[t], *__restrict__ m = a.m[t], *__restrict__ v = a.v[t];
  const float inv_bc1 = a.inv_bc1[t], inv_sqrt_bc2 = a.inv_sqrt_bc2[t];
  auto ld = [](const float* q) {
    return STREAM ? __builtin_nontemporal_load(reinterpret_cast<const adamw_f32x4*>(q))
               : *reinterpret_cast<const adamw_f32x4*>(q);
  };
  auto st = [](adamw_f32x4 x, float* q) {
    if (STREAM) __builtin_nontemporal_store(x, reinterpret_cast<adamw_f32x4*>(q));
    else *reinterpret_cast<adamw_f32x4*>(q) = x;
  };
  bf16x4 gv[ADAMW_UNROLL];
  adamw_f32x4 mw[ADAMW_UNROLL], mv[ADAMW_UNROLL], vv[ADAMW_UNROLL];
#pragma unroll
  for (int u = 0; u < ADAMW_UNROLL; ++u) {
    const long i = i0 + (u * 256 + threadIdx.x) * 4;
    if (i < end) {
      gv[u] = *reinterpret_cast<const bf16x4*>(g + i);
      mw[u] = ld(master + i);
      mv[u] = ld(m + i);
      vv[u] = ld(v + i);
    }
  }
#pragma unroll
  for (int u = 0; u < ADAMW_UNROLL; ++u) {
    const long i = i0 + (u * 256 + threadIdx.x) * 4;
    if (i < end) {
      bf16x4 out;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float gf = bf2f(gv[u].v[j]);
        float w = mw[u][j] * wd_factor;
        const float m_ = b1 * mv[u][j] + (1.f - b1) * gf;
        const float v_ = b2 * vv[u][j] + (1.f - b2) * gf * gf;
        const float denom = sqrtf(v_) * inv_sqrt_bc2 + eps;
        w -= lr * inv_bc1 * m_ / denom;
        mw[u][j] = w; mv[u][j] = m_; vv[u][j] = v_;
        out.v[j] = f2bf(w);
      }
      st(mw[u], master + i);
      st(mv[u], m + i);
      st(vv[u], v + i);
      *reinterpret_cast<bf16x4*>(p + i) = out;
    }
  }
}

// bf16-STATE variant: param/grad/m/v all bf16, NO fp32 master — halves
// optimizer memory for single-GPU 30B-class benches (update math in fp32
// registers; only the stored moments are quantized).
__global__ void adamw_bf16_state_kernel(bf16* __restrict__ p, const bf16* __restrict__ g,
                                        bf16* __restrict__ m, bf16* __restrict__ v,
                                        long n4, float lr, float b1, float b2,
                                        float eps, float wd_factor, float inv_bc1,
                                        float inv_sqrt_bc2) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n4;
       i += (long)gridDim.x * blockDim.x) {
    bf16x4 gv = reinterpret_cast<const bf16x4*>(g)[i];
    bf16x4 pv = reinterpret_cast<const bf16x4*>(p)[i];
    bf16x4 mv = reinterpret_cast<const bf16x4*>(m)[i];
    bf16x4 vv = reinterpret_cast<const bf16x4*>(v)[i];
    bf16x4 pout, mout, vout;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float gf = bf2f(gv.v[j]);
      float w = bf2f(pv.v[j]) * wd_factor;
      float m_ = b1 * bf2f(mv.v[j]) + (1.f - b1) * gf;
      float v_ = b2 * bf2f(vv.v[j]) + (1.f - b2) * gf * gf;
      float denom = sqrtf(v_) * inv_sqrt_bc2 + eps;
      w -= lr * inv_bc1 * m_ / denom;
      mout.v[j] = f2bf(m_); vout.v[j] = f2bf(v_); pout.v[j] = f2bf(w);
    }
    reinterpret_cast<bf16x4*>(m)[i] = mout;
    reinterpret_cast<bf16x4*>(v)[i] = vout;
    reinterpret_cast<bf16x4*>(p)[i] = pout;
  }
}

// fp32-param variant (no separate master copy); grad may be fp32 too.
__global__ void adamw_f32_kernel(float* __restrict__ p, const float* __restrict__ g,
                                 float* __restrict__ m, float* __restrict__ v, long n,
                                 float lr, float b1, float b2, float eps,
                                 float wd_factor, float inv_bc1, float inv_sqrt_bc2) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long)gridDim.x * blockDim.x) {
    float gf = g[i];
    float w = p[i] * wd_factor;
    float m_ = b1 * m[i] + (1.f - b1) * gf;
    float v_ = b2 * v[i] + (1.f - b2) * gf * gf;
    w -= lr * inv_bc1 * m_ / (sqrtf(v_) * inv_sqrt_bc2 + eps);
    p[i] = w; m[i] = m_; v[i] = v_;
  }
}

// bf16 parameters and gradients, f32 master copies and moments, all dense
void adamw_steps(at::TensorList params, at::TensorList grads, at::TensorList masters,
                 at::TensorList ms, at::TensorList vs, at::IntArrayRef steps, double lr,
                 double beta1, double beta2, double eps, double weight_decay) {
  const size_t count = params.size();
  TORCH_CHECK(grads.size() == count && masters.size() == count && ms.size() == count &&
                  vs.size() == count && steps.size() == count,
              "adamw_steps: as many of each");
  auto stream = c10::hip::getCurrentHIPStream();
  AdamwTensors a;
  a.count = 0;
  unsigned blocks = 0;
  long total = 0;
  for (const auto& p : params) total += p.numel();
  auto kernel = total > ADAMW_CACHED ? adamw_bf16_kernel<true> : adamw_bf16_kernel<false>;
  auto launch = [&] {
    if (blocks == 0) return;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, stream.stream(), a, (float)lr,
                       (float)beta1, (float)beta2, (float)eps, (float)(1.0 - lr * weight_decay));
    HIP_CHECK_KERNEL();
    a.count = 0;
    blocks = 0;
  };
  for (size_t t = 0; t < count; ++t) {
    const long n = params[t].numel();
    for (const auto* x : {&params[t], &grads[t]})
      TORCH_CHECK(x->is_cuda() && x->scalar_type() == at::kBFloat16 && x->numel() == n,
                  "adamw_steps: bf16 parameters and gradients on the GPU");
    for (const auto* x : {&masters[t], &ms[t], &vs[t]})
      TORCH_CHECK(x->is_cuda() && x->scalar_type() == at::kFloat && x->numel() == n,
                  "adamw_steps: f32 states on the GPU");
    TORCH_CHECK(n % 4 == 0, "adamw_step: numel must be multiple of 4");
    if (n == 0) continue;
    const unsigned chunks = (unsigned)((n + ADAMW_CHUNK - 1) / ADAMW_CHUNK);
    if (a.count == ADAMW_TENSORS || blocks + chunks > (1u << 22)) launch();
    const int c = a.count++;
    a.p[c] = reinterpret_cast<bf16*>(params[t].data_ptr());
    a.g[c] = reinterpret_cast<const bf16*>(grads[t].data_ptr());
    a.master[c] = masters[t].data_ptr<float>();
    a.m[c] = ms[t].data_ptr<float>();
    a.v[c] = vs[t].data_ptr<float>();
    a.first[c] = blocks;
    a.n[c] = n;
    a.inv_bc1[c] = (float)(1.0 / (1.0 - std::pow(beta1, (double)steps[t])));
    a.inv_sqrt_bc2[c] = (float)(1.0 / std::sqrt(1.0 - std::pow(beta2, (double)steps[t])));
    blocks += chunks;
  }
  launch();
}

void adamw_step(at::Tensor param, at::Tensor grad, at::Tensor master, at::Tensor m,
                at::Tensor v, int64_t step, double lr, double beta1, double beta2,
                double eps, double weight_decay) {
  TORCH_CHECK(param.is_cuda(), "adamw_step: CUDA only");
  const double bc1 = 1.0 - std::pow(beta1, (double)step);
  const double bc2 = 1.0 - std::pow(beta2, (double)step);
  const float wd_factor = (float)(1.0 - lr * weight_decay);
  const float inv_bc1 = (float)(1.0 / bc1);
  const float inv_sqrt_bc2 = (float)(1.0 / std::sqrt(bc2));
  auto stream = c10::hip::getCurrentHIPStream();
  const int block = 256;
  if (param.scalar_type() == at::kBFloat16 && m.scalar_type() == at::kBFloat16) {
    TORCH_CHECK(param.numel() % 4 == 0, "adamw_step: numel must be multiple of 4");
    const long n4 = param.numel() / 4;
    const int grid = (int)std::min<long>((n4 + block - 1) / block, 4096);
    hipLaunchKernelGGL(adamw_bf16_state_kernel, dim3(grid), dim3(block), 0,
                       stream.stream(),
                       reinterpret_cast<bf16*>(param.data_ptr()),
                       reinterpret_cast<const bf16*>(grad.data_ptr()),
                       reinterpret_cast<bf16*>(m.data_ptr()),
                       reinterpret_cast<bf16*>(v.data_ptr()),
                       n4, (float)lr, (float)beta1, (float)beta2, (float)eps,
                       wd_factor, inv_bc1, inv_sqrt_bc2);
  } else if (param.scalar_type() == at::kBFloat16) {
    adamw_steps({param}, {grad}, {master}, {m}, {v}, {step}, lr, beta1, beta2, eps, weight_decay);
    return;
  } else {
    const long n = param.numel();
    const int grid = (int)std::min<long>((n + block - 1) / block, 4096);
    hipLaunchKernelGGL(adamw_f32_kernel, dim3(grid), dim3(block), 0, stream.stream(),
                       param.data_ptr<float>(), grad.data_ptr<float>(),
                       m.data_ptr<float>(), v.data_ptr<float>(), n,
                       (float)lr, (float)beta1, (float)beta2, (float)eps,
                       wd_factor, inv_bc1, inv_sqrt_bc2);
  }
  HIP_CHECK_KERNEL();
}

}  // namespace amd_ops
