// The MoE router's linear layer: bf16 tokens x [T, H] and bf16 weights w [E, H], float32 scores.
//
// A product of two bf16 numbers is exact in float32, so the matrix cores' bf16 products summed in
// float32 are the float32 product of the widened operands; no float32 copy of x is made. Backward,
// the float32 gradient is cut into three bf16 parts of 8 bits each, which hold it exactly, and
// the three products are summed in float32.
//
// Forward and backward read x once (dw once per 64 experts), write dx once and are bound by that,
// and by the latency of the loads at few tokens. us against float32 copies, float32 matrix products and
// copies back to bf16; relative error of the scores against 64 bits on both sides:
//   8192 x 2048, 128 experts: forward 55.5 -> 22.2, backward 132 -> 45 (dx 20, dw 26); 3.9e-7 -> 1.0e-7
//   3003 x 2048,  64 experts: 30.5 -> 9.3 and 69 -> 26; 1.7e-7 -> 1.0e-7
//     60 x 1024,   8 experts: 29 -> 4.9 and 56 -> 12; 1.1e-7 -> 0.8e-7
// dx and dw are off by their rounding to bf16 on both sides (1.66e-3).

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include "common.h"
#include "ops_api.h"

namespace amd_ops {
namespace {

typedef __bf16 rl_bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned rl_u4 __attribute__((ext_vector_type(4)));
typedef float rl_f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ rl_f4 rl_mfma(rl_u4 a, rl_u4 b, rl_f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(rl_bf16x8, a), __builtin_bit_cast(rl_bf16x8, b),
                                                 c, 0, 0, 0);
}

__device__ __forceinline__ rl_u4 rl_load(const bf16* p) { return *reinterpret_cast<const rl_u4*>(p); }

// An 8 x 8 block, row r in rows[r]: column j's eight values are put side by side in cols[j], the
// form in which the matrix core takes eight steps of the contraction from a lane.
__device__ __forceinline__ void rl_transpose(const rl_u4 (&rows)[8], rl_u4 (&cols)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int p = 0; p < 4; ++p)
      cols[j][p] = __builtin_amdgcn_perm(rows[2 * p + 1][j >> 1], rows[2 * p][j >> 1],
                                         j & 1 ? 0x07060302u : 0x05040100u);
}

// v = the sum of three numbers of 8 bits, each the upper half of a float
__device__ __forceinline__ void rl_split(float v, unsigned (&part)[3]) {
  const unsigned hi = __float_as_uint(v) & 0xffff0000u;
  const float r = v - __uint_as_float(hi);
  const bool finite = fabsf(v) < __builtin_inff();
  const unsigned mid = finite ? __float_as_uint(r) & 0xffff0000u : 0u;
  part[0] = v == v ? hi : 0x7fc00000u;
  part[1] = mid;
  part[2] = finite ? __float_as_uint(r - __uint_as_float(mid)) : 0u;
}

__device__ __forceinline__ void rl_split8(const float (&v)[8], rl_u4 (&a)[3]) {
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    unsigned lo[3], hi[3];
    rl_split(v[2 * p], lo);
    rl_split(v[2 * p + 1], hi);
#pragma unroll
    for (int q = 0; q < 3; ++q) a[q][p] = __builtin_amdgcn_perm(hi[q], lo[q], 0x07060302u);
  }
}

// ---- scores[t][e] = sum over h of x[t][h] w[e][h] ----------------------------
// A workgroup of 8 waves takes 32 tokens and 16 NT experts, the waves 64 of every 512 h, a whole
// 128-byte line of a row each: few tokens still have 8 short chains.
template <int NT>
__global__ __launch_bounds__(512) void router_fwd_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                         float* __restrict__ out, int T, int H, int E) {
  constexpr int N = 16 * NT;
  __shared__ float red[4][32 * N];
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63, l = lane & 15, g = lane >> 4;
  const int t0 = blockIdx.x * 32, e0 = blockIdx.y * N;
  const bf16* xr[2];
  const bf16* wr[NT];
#pragma unroll
  for (int m = 0; m < 2; ++m) xr[m] = x + (long)min(t0 + 16 * m + l, T - 1) * H + g * 8;
#pragma unroll
  for (int n = 0; n < NT; ++n) wr[n] = w + (long)min(e0 + 16 * n + l, E - 1) * H + g * 8;
  rl_f4 acc[2][NT] = {};
  for (int h = wid * 64; h < H; h += 512) {
#pragma unroll
    for (int s = 0; s < 64; s += 32) {
      rl_u4 a[2], b[NT];
#pragma unroll
      for (int m = 0; m < 2; ++m) a[m] = rl_load(xr[m] + h + s);
#pragma unroll
      for (int n = 0; n < NT; ++n) b[n] = rl_load(wr[n] + h + s);
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = rl_mfma(a[m], b[n], acc[m][n]);
    }
  }
  // the upper four waves' sums, then the lower four's on top, then the four of each score
  float* mine = red[wid & 3];
#pragma unroll
  for (int half = 1; half >= 0; --half) {
    if (wid >> 2 == half)
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float& r = mine[(16 * m + 4 * g + i) * N + 16 * n + l];
            r = half ? acc[m][n][i] : r + acc[m][n][i];
          }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < 32 * N; i += 512) {
    const int t = t0 + i / N, e = e0 + i % N;
    if (t < T && e < E) out[(long)t * E + e] = (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]);
  }
}

// ---- dx[t][h] = sum over e of d[t][e] w[e][h] --------------------------------
// A wave keeps 128 columns of all (32 KS) experts' weights in registers, transposed once, and walks
// over tiles of 16 tokens; a lane owns 8 neighbouring columns, so nothing passes through LDS.
template <int KS>
__global__ __launch_bounds__(256, 2) void router_dx_kernel(const float* __restrict__ d, const bf16* __restrict__ w,
                                                           bf16* __restrict__ dx, int T, int H, int E) {
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63, l = lane & 15, g = lane >> 4;
  const int h = blockIdx.x * 128 + l * 8;
  rl_u4 b[KS][8];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    rl_u4 rows[8];
    const int e = s * 32 + g * 8;                // E is a multiple of 8
#pragma unroll
    for (int r = 0; r < 8; ++r) rows[r] = e < E ? rl_load(w + (long)(e + r) * H + h) : rl_u4{};
    rl_transpose(rows, b[s]);
  }
  const int tiles = (T + 15) / 16;
  for (int tile = blockIdx.y * 4 + wid; tile < tiles; tile += gridDim.y * 4) {
    const float* dr = d + (long)min(tile * 16 + l, T - 1) * E;
    rl_f4 acc[8] = {};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int e = s * 32 + g * 8;
      rl_f4 v0{}, v1{};
      if (e < E) {
        v0 = *reinterpret_cast<const rl_f4*>(dr + e);
        v1 = *reinterpret_cast<const rl_f4*>(dr + e + 4);
      }
      const float v[8] = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
      rl_u4 a[3];
      rl_split8(v, a);
#pragma unroll
      for (int q = 2; q >= 0; --q)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] = rl_mfma(a[q], b[s][j], acc[j]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = tile * 16 + g * 4 + i;
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o.v[j] = f2bf(acc[j][i]);
      if (t < T) *reinterpret_cast<bf16x8*>(dx + (long)t * H + h) = o;
    }
  }
}

// ---- dw[e][h] = sum over t of d[t][e] x[t][h] --------------------------------
// A wave sums 64 experts by 128 columns over its tokens, 32 at a time, both operands transposed in
// registers; the four waves of a workgroup add up in LDS, and the workgroups' sums, each in a
// place of its own, are added by a second launch in a fixed order.
__global__ __launch_bounds__(256, 2) void router_dw_kernel(const float* __restrict__ d, const bf16* __restrict__ x,
                                                           float* __restrict__ part, int T, int H, int E) {
  __shared__ float red[2][64 * 128];
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63, l = lane & 15, g = lane >> 4;
  const int h = blockIdx.x * 128 + l * 8, e = blockIdx.y * 64 + l * 4;
  rl_f4 acc[4][8] = {};
  for (int t0 = (blockIdx.z * 4 + wid) * 32; t0 < T; t0 += gridDim.z * 128) {
    rl_u4 b[8];
    {
      rl_u4 rows[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const int t = t0 + g * 8 + r;
        rows[r] = t < T ? rl_load(x + (long)t * H + h) : rl_u4{};
      }
      rl_transpose(rows, b);
    }
    rl_f4 dv[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int t = t0 + g * 8 + r;
      dv[r] = t < T && e < E ? *reinterpret_cast<const rl_f4*>(d + (long)t * E + e) : rl_f4{};
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v[8] = {dv[0][i], dv[1][i], dv[2][i], dv[3][i], dv[4][i], dv[5][i], dv[6][i], dv[7][i]};
      rl_u4 a[3];
      rl_split8(v, a);
#pragma unroll
      for (int q = 2; q >= 0; --q)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = rl_mfma(a[q], b[j], acc[i][j]);
    }
  }
  // waves 2 and 3 leave their sums, 0 and 1 add theirs; then all add the two and write
  float* mine = red[wid & 1];
#pragma unroll
  for (int half = 1; half >= 0; --half) {
    if (wid >> 1 == half)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int j = 0; j < 8; j += 4) {
            rl_f4* at = reinterpret_cast<rl_f4*>(mine + ((4 * g + r) * 4 + i) * 128 + l * 8 + j);
            rl_f4 v = {acc[i][j][r], acc[i][j + 1][r], acc[i][j + 2][r], acc[i][j + 3][r]};
            *at = half ? v : *at + v;
          }
    __syncthreads();
  }
  float* dst = part + (long)blockIdx.z * E * H + blockIdx.x * 128;
  for (int i = threadIdx.x; i < 64 * 32; i += 256) {
    const int row = blockIdx.y * 64 + i / 32, c = i % 32 * 4;
    if (row < E)
      *reinterpret_cast<rl_f4*>(dst + (long)row * H + c) =
          *reinterpret_cast<const rl_f4*>(red[0] + i * 4) + *reinterpret_cast<const rl_f4*>(red[1] + i * 4);
  }
}

__global__ __launch_bounds__(256) void router_dw_sum_kernel(const float* __restrict__ part, bf16* __restrict__ dw,
                                                            long n, int splits) {
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;      // n is a multiple of 4
  if (i >= n) return;
  rl_f4 s{};
#pragma unroll 4
  for (int z = 0; z < splits; ++z) s += *reinterpret_cast<const rl_f4*>(part + z * n + i);
  bf16x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) o.v[j] = f2bf(s[j]);
  *reinterpret_cast<bf16x4*>(dw + i) = o;
}

at::Tensor rl_plain(const at::Tensor& t) {      // whole and on a 16-byte boundary
  auto c = t.contiguous();
  return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 ? c.clone() : c;
}

void rl_check(const at::Tensor& x, const at::Tensor& w) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.scalar_type() == at::kBFloat16 && w.device() == x.device() &&
                  w.dim() == 2 && w.scalar_type() == at::kBFloat16 && w.size(1) == x.size(1),
              "router_linear: x [T,H], w [E,H] bfloat16");
  TORCH_CHECK(x.size(1) >= 128 && x.size(1) % 128 == 0 && x.size(1) <= (1 << 20) && w.size(0) >= 8 &&
                  w.size(0) <= 128 && w.size(0) % 8 == 0 && x.size(0) >= 1 && x.size(0) < (1l << 30),
              "router_linear: H in 128s, E in 8s up to 128, at least one token");
}

}  // namespace

at::Tensor router_linear(const at::Tensor& x_, const at::Tensor& w_) {
  rl_check(x_, w_);
  const c10::DeviceGuard guard(x_.device());
  auto x = rl_plain(x_), w = rl_plain(w_);
  const int T = (int)x.size(0), H = (int)x.size(1), E = (int)w.size(0);
  auto out = at::empty({T, E}, x.options().dtype(at::kFloat));
  auto launch = [&](auto kernel, int nt) {
    hipLaunchKernelGGL(kernel, dim3((T + 31) / 32, (E + 16 * nt - 1) / (16 * nt)), dim3(512), 0,
                       c10::hip::getCurrentHIPStream().stream(), (const bf16*)x.data_ptr(),
                       (const bf16*)w.data_ptr(), out.data_ptr<float>(), T, H, E);
  };
  // The fewest experts a workgroup, its chain being short then, that one round of 256 workgroups
  // covers. us at 16, 32, 64, 128 experts a workgroup, 2048 columns: 1000 x 128: 7.3, 9.2, 13.0, 21.0;
  // 2000 x 128: 13.9, 9.6, 13.2, 21.1; 4096 x 128: 23.6, 17.0, 13.7, 21.4; 8192 x 128: 43.9, 30.8,
  // 24.7, 22.5; 65536 x 64: 180, 119, 102, 133.
  int nt = 1;
  while (nt < 8 && 16 * nt < E && (long)((T + 31) / 32) * ((E + 16 * nt - 1) / (16 * nt)) > 256) nt *= 2;
  if (nt == 1) launch(router_fwd_kernel<1>, 1);
  else if (nt == 2) launch(router_fwd_kernel<2>, 2);
  else if (nt == 4) launch(router_fwd_kernel<4>, 4);
  else launch(router_fwd_kernel<8>, 8);
  HIP_CHECK_KERNEL();
  return out;
}

// d [T, E] float32 -> dx [T, H], dw [E, H] bfloat16 (empty where not wanted)
std::tuple<at::Tensor, at::Tensor> router_linear_bwd(const at::Tensor& d_, const at::Tensor& x_,
                                                     const at::Tensor& w_, bool want_dx, bool want_dw) {
  rl_check(x_, w_);
  TORCH_CHECK(d_.device() == x_.device() && d_.dim() == 2 && d_.scalar_type() == at::kFloat &&
                  d_.size(0) == x_.size(0) && d_.size(1) == w_.size(0), "router_linear_bwd: d [T,E] float32");
  const c10::DeviceGuard guard(x_.device());
  auto d = rl_plain(d_);
  const int T = (int)x_.size(0), H = (int)x_.size(1), E = (int)w_.size(0);
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const int cols = H / 128;
  at::Tensor dx, dw;
  if (want_dx) {
    auto w = rl_plain(w_);
    dx = at::empty({T, H}, x_.options());
    // two waves a SIMD: 512 workgroups
    const int groups = std::max(1, std::min((T + 63) / 64, 512 / cols));
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(cols, groups), dim3(256), 0, stream, d.data_ptr<float>(),
                         (const bf16*)w.data_ptr(), (bf16*)dx.data_ptr(), T, H, E);
    };
    if (E <= 32) launch(router_dx_kernel<1>);
    else if (E <= 64) launch(router_dx_kernel<2>);
    else launch(router_dx_kernel<4>);
  } else {
    dx = at::empty({0}, x_.options());
  }
  if (want_dw) {
    auto x = rl_plain(x_);
    const int rows = (E + 63) / 64;
    const int splits = std::max(1, std::min((T + 127) / 128, 512 / (cols * rows)));
    auto part = at::empty({splits, E, H}, d.options());
    dw = at::empty({E, H}, x_.options());
    hipLaunchKernelGGL(router_dw_kernel, dim3(cols, rows, splits), dim3(256), 0, stream, d.data_ptr<float>(),
                       (const bf16*)x.data_ptr(), part.data_ptr<float>(), T, H, E);
    const long n = (long)E * H;
    hipLaunchKernelGGL(router_dw_sum_kernel, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, stream,
                       part.data_ptr<float>(), (bf16*)dw.data_ptr(), n, splits);
  } else {
    dw = at::empty({0}, x_.options());
  }
  HIP_CHECK_KERNEL();
  return {dx, dw};
}

}  // namespace amd_ops
