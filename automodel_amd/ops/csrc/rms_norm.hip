// RMSNorm forward + backward for bf16 rows (CDNA4). Memory-bound: a row stays in the
// registers of the lanes that load it (16 bytes each), so that it is read once.
//
// Rows of up to 2048 take one wave or a part of one (LPR lanes of ITERS vectors), without
// barriers; longer ones, and those beyond 512 where rows are few, a workgroup (at 4096 a wave would hold 8 vectors of each operand
// a lane, too few waves to hide the loads: 74 against 44 us). The backward gives a workgroup a stretch of rows and
// keeps its share of the weight gradient in registers; the shares go to a [blocks, H]
// buffer and a second kernel adds them up in a fixed order. Atomic adds into one row of H
// sums, 1024 deep on each, were the bound before: 263 us for 8192 x 4096, 219 us for
// 6001 x 2048 and 54 us for 256 x 256; now 44, 24 and 12 us with the sum.
//
// Around a norm stands a residual stream: the sum that is normed, and in the backward the
// gradient that reaches the stream by its other way. Both take that operand here, so that
// the sum and the gradients' sum are no passes of their own.

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include "common.h"
#include "ops_api.h"

namespace amd_ops {

namespace {

// sum over the LPR lanes of a row (a wave's part, a wave, or the workgroup of 256)
template <int LPR>
__device__ __forceinline__ float row_sum(float x, float* red) {
  if constexpr (LPR <= 64) {
#pragma unroll
    for (int off = LPR / 2; off > 0; off >>= 1) x += __shfl_xor(x, off);
    return x;
  } else {
    return block_reduce_sum(x, red);
  }
}

// x: [T, H], w: [H] -> y: [T, H], invrms: [T] f32; with ADD of sum = x + delta, which is
// rounded to bf16 and stored first
template <int LPR, int ITERS, bool ADD>
__global__ __launch_bounds__(256) void rms_norm_fwd_kernel(const bf16* __restrict__ x,
                                                           const bf16* __restrict__ delta,
                                                           bf16* __restrict__ sum,
                                                           const bf16* __restrict__ w,
                                                           bf16* __restrict__ y,
                                                           float* __restrict__ invrms, long T, int H,
                                                           float eps) {
  __shared__ float red[4];
  constexpr int ROWS = 256 / LPR;
  const int l = threadIdx.x % LPR;
  const long row = (long)blockIdx.x * ROWS + threadIdx.x / LPR;
  if (LPR <= 64 && row >= T) return;
  const bf16* xr = x + row * H;
  bf16x8 xv[ITERS];
  float ss = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int i = (l + it * LPR) * 8;
    if (i < H) xv[it] = *reinterpret_cast<const bf16x8*>(xr + i);
  }
  if constexpr (ADD) {
    bf16x8 dv[ITERS];
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int i = (l + it * LPR) * 8;
      if (i < H) dv[it] = *reinterpret_cast<const bf16x8*>(delta + row * H + i);
    }
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int i = (l + it * LPR) * 8;
      if (i < H) {
#pragma unroll
        for (int j = 0; j < 8; ++j) xv[it].v[j] = f2bf(bf2f(xv[it].v[j]) + bf2f(dv[it].v[j]));
        *reinterpret_cast<bf16x8*>(sum + row * H + i) = xv[it];
      }
    }
  }
#pragma unroll
  for (int it = 0; it < ITERS; ++it)
    if ((l + it * LPR) * 8 < H) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float f = bf2f(xv[it].v[j]);
        ss = fmaf(f, f, ss);
      }
    }
  ss = row_sum<LPR>(ss, red);
  const float inv = rsqrtf(ss / (float)H + eps);
  if (l == 0) invrms[row] = inv;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int i = (l + it * LPR) * 8;
    if (i < H) {
      const bf16x8 wv = *reinterpret_cast<const bf16x8*>(w + i);
      bf16x8 out;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        // torch's rounding: x * inv to bf16, then a bf16 product with w
        const float xn = bf2f(f2bf(bf2f(xv[it].v[j]) * inv));
        out.v[j] = f2bf(xn * bf2f(wv.v[j]));
      }
      *reinterpret_cast<bf16x8*>(y + row * H + i) = out;
    }
  }
}

// rows too long for registers: read twice
__global__ __launch_bounds__(256) void rms_norm_fwd_long_kernel(const bf16* __restrict__ x,
                                                                const bf16* __restrict__ w,
                                                                bf16* __restrict__ y,
                                                                float* __restrict__ invrms, int H,
                                                                float eps) {
  __shared__ float red[4];
  const long row = blockIdx.x;
  float ss = 0.f;
  for (int i = threadIdx.x * 8; i < H; i += 256 * 8) {
    const bf16x8 xv = *reinterpret_cast<const bf16x8*>(x + row * H + i);
#pragma unroll
    for (int j = 0; j < 8; ++j) ss = fmaf(bf2f(xv.v[j]), bf2f(xv.v[j]), ss);
  }
  const float inv = rsqrtf(block_reduce_sum(ss, red) / (float)H + eps);
  if (threadIdx.x == 0) invrms[row] = inv;
  for (int i = threadIdx.x * 8; i < H; i += 256 * 8) {
    const bf16x8 xv = *reinterpret_cast<const bf16x8*>(x + row * H + i);
    const bf16x8 wv = *reinterpret_cast<const bf16x8*>(w + i);
    bf16x8 out;
#pragma unroll
    for (int j = 0; j < 8; ++j) out.v[j] = f2bf(bf2f(f2bf(bf2f(xv.v[j]) * inv)) * bf2f(wv.v[j]));
    *reinterpret_cast<bf16x8*>(y + row * H + i) = out;
  }
}

// dx_i = inv * dy_i*w_i - x_i * inv^3 / H * sum_j(dy_j*w_j*x_j) + dres_i
// part[block][i] = sum over the block's rows of dy_i * x_i * inv
// dres (the other gradient of x) and part (wanted weight gradient) may be null
template <int LPR, int ITERS>
__global__ __launch_bounds__(256) void rms_norm_bwd_kernel(const bf16* __restrict__ dy,
                                                           const bf16* __restrict__ x,
                                                           const bf16* __restrict__ w,
                                                           const float* __restrict__ invrms,
                                                           const bf16* __restrict__ dres,
                                                           bf16* __restrict__ dx,
                                                           float* __restrict__ part, long T, int H) {
  constexpr int ROWS = 256 / LPR;      // rows at a time
  __shared__ float red[4];
  __shared__ __attribute__((aligned(16))) float sums[LPR <= 64 ? 4 * 512 : 4];
  const int l = threadIdx.x % LPR;
  float dw[ITERS][8];
#pragma unroll
  for (int it = 0; it < ITERS; ++it)
#pragma unroll
    for (int j = 0; j < 8; ++j) dw[it][j] = 0.f;

  for (long row = (long)blockIdx.x * ROWS + threadIdx.x / LPR; row < T; row += (long)gridDim.x * ROWS) {
    const float inv = invrms[row];
    bf16x8 xv[ITERS], dv[ITERS], rv[ITERS];
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int i = (l + it * LPR) * 8;
      rv[it] = bf16x8{};
      if (i < H) {
        if (dres) rv[it] = *reinterpret_cast<const bf16x8*>(dres + row * H + i);
        xv[it] = *reinterpret_cast<const bf16x8*>(x + row * H + i);
        dv[it] = *reinterpret_cast<const bf16x8*>(dy + row * H + i);
      }
    }
    float s = 0.f;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int i = (l + it * LPR) * 8;
      if (i < H) {
        const bf16x8 wv = *reinterpret_cast<const bf16x8*>(w + i);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float xf = bf2f(xv[it].v[j]), df = bf2f(dv[it].v[j]);
          s = fmaf(df * bf2f(wv.v[j]), xf, s);
          dw[it][j] = fmaf(df, xf * inv, dw[it][j]);
        }
      }
    }
    s = row_sum<LPR>(s, red);
    const float c = s * inv * inv * inv / (float)H;
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int i = (l + it * LPR) * 8;
      if (i < H) {
        const bf16x8 wv = *reinterpret_cast<const bf16x8*>(w + i);
        bf16x8 out;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          out.v[j] = f2bf(inv * bf2f(dv[it].v[j]) * bf2f(wv.v[j]) - bf2f(xv[it].v[j]) * c +
                          bf2f(rv[it].v[j]));
        *reinterpret_cast<bf16x8*>(dx + row * H + i) = out;
      }
    }
  }

  if (!part) return;
  // the block's sums: over the wave's parts by shuffles, over the waves in LDS
  float* to = part + (long)blockIdx.x * H;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int i = (l + it * LPR) * 8;
    if constexpr (LPR <= 64) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int off = LPR; off < 64; off <<= 1) dw[it][j] += __shfl_xor(dw[it][j], off);
      const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
      if (it > 0) __syncthreads();
      if (lane < LPR)
#pragma unroll
        for (int j = 0; j < 8; ++j) sums[wid * 512 + lane * 8 + j] = dw[it][j];
      __syncthreads();
      for (int q = threadIdx.x; q < LPR * 8; q += 256) {
        const int col = it * LPR * 8 + q;
        if (col < H) to[col] = sums[q] + sums[512 + q] + sums[1024 + q] + sums[1536 + q];
      }
    } else if (i < H) {
#pragma unroll
      for (int j = 0; j < 8; ++j) to[i + j] = dw[it][j];
    }
  }
}

// dw[i] = sum over blocks of part[block][i]: 64 columns a workgroup, 16 rows at a time
__global__ __launch_bounds__(256) void rms_norm_dw_kernel(const float* __restrict__ part,
                                                          bf16* __restrict__ dw, int blocks, int H) {
  __shared__ __attribute__((aligned(16))) float4 sums[256];
  const int col = blockIdx.x * 64 + (threadIdx.x & 15) * 4;
  float4 s = {0.f, 0.f, 0.f, 0.f};
  if (col < H)      // H is a multiple of 8
#pragma unroll 4
    for (int r = threadIdx.x >> 4; r < blocks; r += 16) {
      const float4 p = *reinterpret_cast<const float4*>(part + (long)r * H + col);
      s.x += p.x; s.y += p.y; s.z += p.z; s.w += p.w;
    }
  sums[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x < 16 && col < H) {
    for (int r = 1; r < 16; ++r) {
      const float4 p = sums[r * 16 + threadIdx.x];
      s.x += p.x; s.y += p.y; s.z += p.z; s.w += p.w;
    }
    bf16x4 out;
    out.v[0] = f2bf(s.x); out.v[1] = f2bf(s.y); out.v[2] = f2bf(s.z); out.v[3] = f2bf(s.w);
    *reinterpret_cast<bf16x4*>(dw + col) = out;
  }
}

// calls f(lanes per row, vectors per lane) for T rows of H. A row of more than 512 columns
// takes one wave where that gives the chip enough of them, and the workgroup where there are
// few: then the row's own chain of two or four loads and sums a lane is the time (us, a
// wave's row against a workgroup's)
//                     1 row  64    256   1000  2000  4096
//   2048, forward     3.0    3.7   3.8   4.2   4.8   6.9
//                     2.3    2.8   2.8   3.4   4.5   7.0
//   2048, backward    6.7    7.6   7.9   10.8  14.0  19.2
//                     4.8    5.4   7.3   15.7  16.9  20.7
//   768, forward      2.5    2.9   2.9   3.0   3.3   4.1
//                     2.4    2.7   2.8   3.0   3.6   5.3
//   768, backward     5.3    5.7   6.0   8.1   9.9   11.1
//                     4.8    5.2   6.6   12.8  13.5  15.8
// The lines cross at about as many rows as columns, and in the backward at an eighth of
// that: a workgroup's share of the weight gradient is a row of sums for each row then.
template <typename F>
void by_row_size(long T, int H, long few, F f) {
  using std::integral_constant;
#define RMS_CASE(MAX, LPR, ITERS) \
  if (H <= MAX) return f(integral_constant<int, LPR>{}, integral_constant<int, ITERS>{});
  RMS_CASE(128, 16, 1)
  RMS_CASE(256, 32, 1)
  RMS_CASE(512, 64, 1)
  if (H <= 2048 && T <= few)
    return f(integral_constant<int, 256>{}, integral_constant<int, 1>{});
  RMS_CASE(1024, 64, 2)
  RMS_CASE(2048, 64, 4)
  RMS_CASE(4096, 256, 2)
  RMS_CASE(8192, 256, 4)
  RMS_CASE(16384, 256, 8)
#undef RMS_CASE
  TORCH_CHECK(false, "rms_norm_bwd: H too large: ", H);
}

constexpr int MAX_IN_REGISTERS = 16384;

}  // namespace

namespace {

const bf16* data(const at::Tensor& t) { return reinterpret_cast<const bf16*>(t.data_ptr()); }
bf16* out(const at::Tensor& t) { return reinterpret_cast<bf16*>(t.data_ptr()); }

template <bool ADD>
void launch_fwd(const at::Tensor& x, const bf16* delta, bf16* sum, const at::Tensor& w,
                const at::Tensor& y, const at::Tensor& invrms, double eps) {
  const long T = x.size(0);
  const int H = x.size(1);
  by_row_size(T, H, H, [&](auto lpr, auto iters) {
    constexpr int LPR = lpr.value, ITERS = iters.value;
    hipLaunchKernelGGL((rms_norm_fwd_kernel<LPR, ITERS, ADD>), dim3(ceil_div_i(T, 256 / LPR)),
                       dim3(256), 0, c10::hip::getCurrentHIPStream().stream(), data(x), delta, sum,
                       data(w), out(y), invrms.data_ptr<float>(), T, H, (float)eps);
  });
  HIP_CHECK_KERNEL();
}

}  // namespace

std::tuple<at::Tensor, at::Tensor> rms_norm_fwd(const at::Tensor& x,
                                                const at::Tensor& w,
                                                double eps) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.scalar_type() == at::kBFloat16,
              "rms_norm_fwd: x must be 2-D bf16 CUDA");
  const long T = x.size(0);
  const int H = x.size(1);
  TORCH_CHECK(H % 8 == 0, "rms_norm_fwd: H must be a multiple of 8, got ", H);
  auto y = at::empty_like(x);
  auto invrms = at::empty({T}, x.options().dtype(at::kFloat));
  if (H > MAX_IN_REGISTERS) {
    hipLaunchKernelGGL(rms_norm_fwd_long_kernel, dim3(T), dim3(256), 0,
                       c10::hip::getCurrentHIPStream().stream(), data(x), data(w), out(y),
                       invrms.data_ptr<float>(), H, (float)eps);
    HIP_CHECK_KERNEL();
    return {y, invrms};
  }
  launch_fwd<false>(x, nullptr, nullptr, w, y, invrms, eps);
  return {y, invrms};
}

// -> x + delta, its norm, invrms
std::tuple<at::Tensor, at::Tensor, at::Tensor> add_rms_norm_fwd(const at::Tensor& x,
                                                                const at::Tensor& delta,
                                                                const at::Tensor& w, double eps) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.scalar_type() == at::kBFloat16 &&
                  x.is_contiguous() && x.size(0) >= 1,
              "add_rms_norm_fwd: x [T, H] bf16");
  TORCH_CHECK(delta.device() == x.device() && delta.sizes() == x.sizes() &&
                  delta.scalar_type() == at::kBFloat16 && delta.is_contiguous(),
              "add_rms_norm_fwd: delta as x");
  TORCH_CHECK(w.device() == x.device() && w.scalar_type() == at::kBFloat16 && w.dim() == 1 &&
                  w.size(0) == x.size(1) && w.is_contiguous() && x.size(1) % 8 == 0 &&
                  x.size(1) <= MAX_IN_REGISTERS,
              "add_rms_norm_fwd: w [H] bf16, H a multiple of 8 and at most ", MAX_IN_REGISTERS);
  auto sum = at::empty_like(x), y = at::empty_like(x);
  auto invrms = at::empty({x.size(0)}, x.options().dtype(at::kFloat));
  launch_fwd<true>(x, data(delta), out(sum), w, y, invrms, eps);
  return {sum, y, invrms};
}

// -> dx (+ dres), dw (undefined if it is not wanted)
std::tuple<at::Tensor, at::Tensor> rms_norm_bwd(const at::Tensor& dy,
                                                const at::Tensor& x,
                                                const at::Tensor& w,
                                                const at::Tensor& invrms,
                                                const std::optional<at::Tensor>& dres,
                                                bool want_dw) {
  const long T = x.size(0);
  const int H = x.size(1);
  TORCH_CHECK(!dres || (dres->device() == x.device() && dres->sizes() == x.sizes() &&
                        dres->scalar_type() == at::kBFloat16 && dres->is_contiguous()),
              "rms_norm_bwd: dres as x");
  auto dx = at::empty_like(x);
  at::Tensor dw, part;
  auto stream = c10::hip::getCurrentHIPStream().stream();
  by_row_size(T, H, H / 8, [&](auto lpr, auto iters) {
    constexpr int LPR = lpr.value, ITERS = iters.value;
    // enough workgroups to fill the chip; more only add to the sums that are written and
    // read again (8192 x 4096: 52 us with 512, 44 with 1024, 53 with 2048; 6001 x 2048,
    // where a wave has a row of its own: 28 with 256, 24 with 512, 29 with 1024)
    const int blocks = (int)std::min<long>((T + 256 / LPR - 1) / (256 / LPR), LPR > 64 ? 1024 : 512);
    if (want_dw) {
      dw = at::empty({H}, x.options());
      part = at::empty({blocks, H}, x.options().dtype(at::kFloat));
    }
    hipLaunchKernelGGL((rms_norm_bwd_kernel<LPR, ITERS>), dim3(blocks), dim3(256), 0, stream,
                       data(dy), data(x), data(w), invrms.data_ptr<float>(),
                       dres ? data(*dres) : nullptr, out(dx),
                       want_dw ? part.data_ptr<float>() : nullptr, T, H);
    if (want_dw)
      hipLaunchKernelGGL(rms_norm_dw_kernel, dim3(ceil_div_i(H, 64)), dim3(256), 0, stream,
                         part.data_ptr<float>(), out(dw), blocks, H);
  });
  HIP_CHECK_KERNEL();
  return {dx, dw};
}

}  // namespace amd_ops
