// Fused SwiGLU elementwise kernels: y = silu(g) * u, plus backward.
// Memory-bound; bf16x8 vector loads, grid-stride (guide Guideline 11/13).

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include "common.h"
#include "ops_api.h"

namespace amd_ops {

__device__ __forceinline__ float sigmoidf_(float x) { return 1.f / (1.f + __expf(-x)); }

__global__ void swiglu_fwd_kernel(const bf16* __restrict__ g, const bf16* __restrict__ u,
                                  bf16* __restrict__ y, long n8) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n8;
       i += (long)gridDim.x * blockDim.x) {
    bf16x8 gv = reinterpret_cast<const bf16x8*>(g)[i];
    bf16x8 uv = reinterpret_cast<const bf16x8*>(u)[i];
    bf16x8 out;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float gf = bf2f(gv.v[j]);
      out.v[j] = f2bf(gf * sigmoidf_(gf) * bf2f(uv.v[j]));
    }
    reinterpret_cast<bf16x8*>(y)[i] = out;
  }
}

__global__ void swiglu_bwd_kernel(const bf16* __restrict__ dy, const bf16* __restrict__ g,
                                  const bf16* __restrict__ u, bf16* __restrict__ dg,
                                  bf16* __restrict__ du, long n8) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n8;
       i += (long)gridDim.x * blockDim.x) {
    bf16x8 dv = reinterpret_cast<const bf16x8*>(dy)[i];
    bf16x8 gv = reinterpret_cast<const bf16x8*>(g)[i];
    bf16x8 uv = reinterpret_cast<const bf16x8*>(u)[i];
    bf16x8 dgo, duo;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float d = bf2f(dv.v[j]);
      float gf = bf2f(gv.v[j]);
      float uf = bf2f(uv.v[j]);
      float sg = sigmoidf_(gf);
      float silu = gf * sg;
      dgo.v[j] = f2bf(d * uf * sg * (1.f + gf * (1.f - sg)));
      duo.v[j] = f2bf(d * silu);
    }
    reinterpret_cast<bf16x8*>(dg)[i] = dgo;
    reinterpret_cast<bf16x8*>(du)[i] = duo;
  }
}

at::Tensor swiglu_fwd(const at::Tensor& g, const at::Tensor& u) {
  TORCH_CHECK(g.is_cuda() && g.scalar_type() == at::kBFloat16, "swiglu: bf16 CUDA only");
  TORCH_CHECK(g.numel() % 8 == 0, "swiglu: numel must be a multiple of 8");
  auto y = at::empty_like(g);
  const long n8 = g.numel() / 8;
  const int block = 256;
  const int grid = (int)std::min<long>((n8 + block - 1) / block, 2048);
  auto stream = c10::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(swiglu_fwd_kernel, dim3(grid), dim3(block), 0, stream.stream(),
                     reinterpret_cast<const bf16*>(g.data_ptr()),
                     reinterpret_cast<const bf16*>(u.data_ptr()),
                     reinterpret_cast<bf16*>(y.data_ptr()), n8);
  HIP_CHECK_KERNEL();
  return y;
}

std::tuple<at::Tensor, at::Tensor> swiglu_bwd(const at::Tensor& dy, const at::Tensor& g,
                                              const at::Tensor& u) {
  auto dg = at::empty_like(g);
  auto du = at::empty_like(u);
  const long n8 = g.numel() / 8;
  const int block = 256;
  const int grid = (int)std::min<long>((n8 + block - 1) / block, 2048);
  auto stream = c10::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(swiglu_bwd_kernel, dim3(grid), dim3(block), 0, stream.stream(),
                     reinterpret_cast<const bf16*>(dy.data_ptr()),
                     reinterpret_cast<const bf16*>(g.data_ptr()),
                     reinterpret_cast<const bf16*>(u.data_ptr()),
                     reinterpret_cast<bf16*>(dg.data_ptr()),
                     reinterpret_cast<bf16*>(du.data_ptr()), n8);
  HIP_CHECK_KERNEL();
  return {dg, du};
}

// The backward of rows that enter a sum with a weight, out[t] = sum_i p[i] (h[i] w): of the unweighted rows' gradient dh
// the weighted dg and du, p h, which is the operand of w's gradient, and the weights' own, dp[order[i]] = sum(dh[i] h[i]):
// with the products of the sum, out is not needed again. 32 lanes a row, so that rows of 768 and 1408 columns leave few
// of them idle. Bound by its six passes over a row: 65536 x 768 98 us, 6.2 TB/s (with combine_bwd and swiglu_bwd that it stands
// for 215 us, here with the copies of the rows 145)
__global__ __launch_bounds__(256) void swiglu_rows_bwd_kernel(const bf16* __restrict__ dh, const bf16* __restrict__ g,
                                                              const bf16* __restrict__ u, const float* __restrict__ p,
                                                              const int* __restrict__ order, bf16* __restrict__ dg,
                                                              bf16* __restrict__ du, bf16* __restrict__ ph,
                                                              float* __restrict__ dp, long M, int I) {
  const long row = (long)blockIdx.x * 8 + (threadIdx.x >> 5);
  if (row >= M) return;
  const int lane = threadIdx.x & 31;
  const float w = p[row];
  float s = 0.f;
#pragma unroll 3
  for (int c = lane * 8; c < I; c += 256) {
    const long at = row * I + c;
    const bf16x8 dv = *reinterpret_cast<const bf16x8*>(dh + at), gv = *reinterpret_cast<const bf16x8*>(g + at),
                 uv = *reinterpret_cast<const bf16x8*>(u + at);
    bf16x8 dgo, duo, pho;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float d = bf2f(dv.v[j]), gf = bf2f(gv.v[j]), uf = bf2f(uv.v[j]);
      const float sg = sigmoidf_(gf), silu = gf * sg, h = silu * uf, dw = d * w;
      s = fmaf(d, h, s);
      pho.v[j] = f2bf(w * h);
      dgo.v[j] = f2bf(dw * uf * sg * (1.f + gf * (1.f - sg)));
      duo.v[j] = f2bf(dw * silu);
    }
    *reinterpret_cast<bf16x8*>(dg + at) = dgo;
    *reinterpret_cast<bf16x8*>(du + at) = duo;
    *reinterpret_cast<bf16x8*>(ph + at) = pho;
  }
#pragma unroll
  for (int off = 16; off > 0; off >>= 1) s += __shfl_xor(s, off);
  if (lane == 0) dp[order[row]] = s;
}

// dh, g, u [M, I]; p f32, order int32 [M] -> {dg, du, p h, dp [M]}
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> swiglu_rows_bwd(const at::Tensor& dh, const at::Tensor& g,
                                                                           const at::Tensor& u, const at::Tensor& p,
                                                                           const at::Tensor& order) {
  for (const at::Tensor* t : {&dh, &g, &u})
    TORCH_CHECK(t->is_cuda() && t->device() == dh.device() && t->scalar_type() == at::kBFloat16 && t->dim() == 2 &&
                    t->is_contiguous() && t->sizes() == dh.sizes() && (uintptr_t)t->data_ptr() % 16 == 0 && t->size(1) % 8 == 0,
                "swiglu_rows_bwd: three bf16 [M, I], I%8==0");
  const long M = dh.size(0);
  TORCH_CHECK(p.device() == dh.device() && p.scalar_type() == at::kFloat && p.is_contiguous() && p.numel() == M &&
                  order.device() == dh.device() && order.scalar_type() == at::kInt && order.is_contiguous() &&
                  order.numel() == M && M < (1l << 31), "swiglu_rows_bwd: p float32, order int32 [M]");
  auto dg = at::empty_like(g), du = at::empty_like(g), ph = at::empty_like(g);
  auto dp = at::empty({M}, p.options());
  if (dh.numel() == 0) return {dg, du, ph, dp.zero_()};
  hipLaunchKernelGGL(swiglu_rows_bwd_kernel, dim3((unsigned)((M + 7) / 8)), dim3(256), 0,
                     c10::hip::getCurrentHIPStream().stream(), reinterpret_cast<const bf16*>(dh.data_ptr()),
                     reinterpret_cast<const bf16*>(g.data_ptr()), reinterpret_cast<const bf16*>(u.data_ptr()),
                     p.data_ptr<float>(), order.data_ptr<int>(), reinterpret_cast<bf16*>(dg.data_ptr()),
                     reinterpret_cast<bf16*>(du.data_ptr()), reinterpret_cast<bf16*>(ph.data_ptr()), dp.data_ptr<float>(),
                     M, (int)dh.size(1));
  HIP_CHECK_KERNEL();
  return {dg, du, ph, dp};
}

// Variants over a CONCATENATED [T, 2I] gate|up tensor (fused gate_up_proj
// GEMM output): y[t, i] = silu(gu[t, i]) * gu[t, I + i].
__global__ void swiglu_cat_fwd_kernel(const bf16* __restrict__ gu, bf16* __restrict__ y,
                                      long T, int I) {
  const long t = blockIdx.y;
  const bf16* g = gu + t * (long)(2 * I);
  const bf16* u = g + I;
  bf16* yr = y + t * (long)I;
  for (int i = (blockIdx.x * blockDim.x + threadIdx.x) * 8; i < I;
       i += gridDim.x * blockDim.x * 8) {
    bf16x8 gv = *reinterpret_cast<const bf16x8*>(g + i);
    bf16x8 uv = *reinterpret_cast<const bf16x8*>(u + i);
    bf16x8 out;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float gf = bf2f(gv.v[j]);
      out.v[j] = f2bf(gf * sigmoidf_(gf) * bf2f(uv.v[j]));
    }
    *reinterpret_cast<bf16x8*>(yr + i) = out;
  }
}

__global__ void swiglu_cat_bwd_kernel(const bf16* __restrict__ dy,
                                      const bf16* __restrict__ gu,
                                      bf16* __restrict__ dgu, long T, int I) {
  const long t = blockIdx.y;
  const bf16* g = gu + t * (long)(2 * I);
  const bf16* u = g + I;
  const bf16* d = dy + t * (long)I;
  bf16* dg = dgu + t * (long)(2 * I);
  bf16* du = dg + I;
  for (int i = (blockIdx.x * blockDim.x + threadIdx.x) * 8; i < I;
       i += gridDim.x * blockDim.x * 8) {
    bf16x8 dv = *reinterpret_cast<const bf16x8*>(d + i);
    bf16x8 gv = *reinterpret_cast<const bf16x8*>(g + i);
    bf16x8 uv = *reinterpret_cast<const bf16x8*>(u + i);
    bf16x8 dgo, duo;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float dd = bf2f(dv.v[j]);
      float gf = bf2f(gv.v[j]);
      float uf = bf2f(uv.v[j]);
      float sg = sigmoidf_(gf);
      dgo.v[j] = f2bf(dd * uf * sg * (1.f + gf * (1.f - sg)));
      duo.v[j] = f2bf(dd * gf * sg);
    }
    *reinterpret_cast<bf16x8*>(dg + i) = dgo;
    *reinterpret_cast<bf16x8*>(du + i) = duo;
  }
}

at::Tensor swiglu_cat_fwd(const at::Tensor& gu) {
  TORCH_CHECK(gu.is_cuda() && gu.scalar_type() == at::kBFloat16 && gu.dim() == 2,
              "swiglu_cat: [T, 2I] bf16");
  const long T = gu.size(0);
  const int I = gu.size(1) / 2;
  TORCH_CHECK(I % 8 == 0, "swiglu_cat: I % 8 == 0");
  auto y = at::empty({T, (long)I}, gu.options());
  const int block = 256;
  const int gx = std::min(32, (I / 8 + block - 1) / block);
  auto stream = c10::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(swiglu_cat_fwd_kernel, dim3(gx, T), dim3(block), 0, stream.stream(),
                     reinterpret_cast<const bf16*>(gu.data_ptr()),
                     reinterpret_cast<bf16*>(y.data_ptr()), T, I);
  HIP_CHECK_KERNEL();
  return y;
}

at::Tensor swiglu_cat_bwd(const at::Tensor& dy, const at::Tensor& gu) {
  const long T = gu.size(0);
  const int I = gu.size(1) / 2;
  auto dgu = at::empty_like(gu);
  const int block = 256;
  const int gx = std::min(32, (I / 8 + block - 1) / block);
  auto stream = c10::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(swiglu_cat_bwd_kernel, dim3(gx, T), dim3(block), 0, stream.stream(),
                     reinterpret_cast<const bf16*>(dy.data_ptr()),
                     reinterpret_cast<const bf16*>(gu.data_ptr()),
                     reinterpret_cast<bf16*>(dgu.data_ptr()), T, I);
  HIP_CHECK_KERNEL();
  return dgu;
}

}  // namespace amd_ops
