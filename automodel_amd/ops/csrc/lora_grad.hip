// Gradients of y = x w^T + scale (x A^T) B^T (gfx950): x [M, H], A [r, H], B [O, r], r a multiple of 8 up to 64,
// filled up to R = 32 or 64 with zeros; t = x A^T is the forward's.
//
//   dt = scale g B        lora_down_kernel (lora.hip) of g and B^T
//   dB = scale g^T t      lora_outer_kernel
//   dA = dt^T x           the same
//   dx = g w + dt A       linear_grad.hip's tiles, dt A behind their sums
//
// All but the last are bound by reading g or x once each. Without dx, us, with the library's products and their
// scalings before: 8192 rows, 4096 -> 6144 118, now 67; 4096 -> 28672 250, now 208 (at 4.82 TB/s: 209);
// 14336 -> 4096 197, now 88; 200 rows, 512 -> 512 26, now 18 (86 on the host, now 18).
#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include "common.h"
#include "linear_tiles.h"
#include "ops_api.h"

namespace amd_ops {

namespace lg {

void launch_extra(const Args& a, unsigned blocks, hipStream_t stream) {
  const auto launch = [&](auto short_, auto parts_) {
    hipLaunchKernelGGL((linear_tile_kernel<DX, decltype(short_)::value, decltype(parts_)::value, true>), dim3(blocks),
                       dim3(gt::THREADS), gt::SMEM, stream, a);
    HIP_CHECK_KERNEL();
  };
  if (a.parts > 1) launch(std::false_type{}, std::true_type{});
  else if (a.sum == 2 * gt::STEP) launch(std::true_type{}, std::false_type{});
  else launch(std::false_type{}, std::false_type{});
}

}  // namespace lg

namespace {

struct Outer {
  const bf16 *x, *y;         // [M, C]; [R, pitch], a row of summed index, zeros from M on
  bf16* out;                 // [C, r], or ACROSS: [r, C]
  float* part;               // [parts][out], of more than one part
  int M, C, pitch, r, per, parts;
  float scale;
};

constexpr int STRIP = 256;   // columns of x of a workgroup

// out = scale sum_m x[m, c] y[r, m]. A workgroup takes 256 columns and a stretch of the rows, 64 of them at a time
// (33 KB of x, two of them in flight; two workgroups share a CU), its waves 64 columns each; 64 rows are two matrix
// instructions for 16 columns x 16 of R, the transposed operand read by LDS's transposing reads. 8192 x 28672:
// 86 us, 5.5 TB/s.
template <int R, bool ACROSS>
__global__ __launch_bounds__(256, 2) void lora_outer_kernel(const Outer a) {
  constexpr int PAIR = 32768 + R * 128, LOADS = 8 + R / 32;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int strips = (a.C + STRIP - 1) / STRIP, c0 = blockIdx.x % strips * STRIP, part = blockIdx.x / strips;
  const int m0 = part * a.per, rows = min(a.per, a.M - m0), n = (rows + 63) / 64;
  gt::Operand<true, true> X;
  gt::Operand<false, true> Y;
  X.init(2u * a.C, wid);
  Y.init(2u * a.pitch, wid);
  X.aim(a.x + (long)m0 * a.C + c0, a.C - c0, rows);
  Y.aim(a.y + m0, R, rows);
  const unsigned lds = fa::lds_address(smem);
  auto load = [&](int p) __attribute__((always_inline)) {
    const unsigned to = lds + p * PAIR + wid * 1024;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int h = 0; h < 4; ++h) gt::load_lds(to, s * 16384 + h * 4096, X.off[h], X.base, X.num);
      X.seek();
    }
#pragma unroll
    for (int h = 0; h < R / 32; ++h) gt::load_lds(to, 32768 + h * 4096, Y.off[h], Y.base, Y.num);
    Y.seek();
  };
  gt::f32x4_t acc[4][R / 16];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < R / 16; ++j) acc[i][j] = gt::f32x4_t{0.f, 0.f, 0.f, 0.f};
  load(0);
  load(1);
#pragma unroll 1
  for (int p = 0; p < n; ++p) {
    const int at = p & 1;
    X.look(lds + at * PAIR, wid * 4);
    Y.look(lds + at * PAIR + 32768, 0);
    fa::wait_loads<LOADS>();
    fa::barrier();
    __builtin_amdgcn_sched_barrier(0);
    fa::unrolled<2>([&](auto s_) __attribute__((always_inline)) {
      constexpr int S = decltype(s_)::value;
      gt::bf16x8_t xf[4], yf[R / 16];
#pragma unroll
      for (int i = 0; i < 4; ++i) X.template read<S>(xf[i], i, 2);
#pragma unroll
      for (int j = 0; j < R / 16; ++j) Y.template read<S>(yf[j], j, 2);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < R / 16; ++j)
          acc[i][j] = ACROSS ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[i], yf[j], acc[i][j], 0, 0, 0)
                             : __builtin_amdgcn_mfma_f32_16x16x32_bf16(yf[j], xf[i], acc[i][j], 0, 0, 0);
    });
    __builtin_amdgcn_sched_barrier(0);
    fa::barrier();
    load(at);
  }
  fa::wait_loads();
  // a lane has 4 of R of one column, or ACROSS 4 columns of one of R
  const int i16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < R / 16; ++j) {
      const int c = c0 + wid * 64 + i * 16;        // C is a multiple of 16
      if (c >= a.C || j * 16 + (ACROSS ? i16 : g * 4) >= a.r) continue;
      const long o = ACROSS ? (long)(j * 16 + i16) * a.C + c + g * 4 : (long)(c + i16) * a.r + j * 16 + g * 4;
      if (a.parts > 1) {
        *reinterpret_cast<gt::f32x4_t*>(a.part + (long)part * a.C * a.r + o) = acc[i][j];
      } else {
        gt::bf16x4_t w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = (__bf16)(acc[i][j][e] * a.scale);
        *reinterpret_cast<gt::bf16x4_t*>(a.out + o) = w;
      }
    }
}

__global__ __launch_bounds__(256) void add_outer_kernel(const float* __restrict__ part, bf16* __restrict__ out, long n,
                                                        int parts, float scale) {
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  gt::f32x4_t s = *reinterpret_cast<const gt::f32x4_t*>(part + i);
#pragma unroll 4
  for (int k = 1; k < parts; ++k) s += *reinterpret_cast<const gt::f32x4_t*>(part + k * n + i);
  gt::bf16x4_t w;
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] = (__bf16)(s[e] * scale);
  *reinterpret_cast<gt::bf16x4_t*>(out + i) = w;
}

// A [r, H] -> [H, R] and B [O, r] -> [R, O], 64 of the long side a workgroup
template <int R>
__global__ __launch_bounds__(256) void turn_kernel(const bf16* __restrict__ A, const bf16* __restrict__ B,
                                                   bf16* __restrict__ At, bf16* __restrict__ Bt, int H, int O,
                                                   int r) {
  __shared__ bf16 s[64][R + 2];
  const int blocks = H / 64;
  const bool a = (int)blockIdx.x < blocks;
  const long at = (a ? blockIdx.x : blockIdx.x - blocks) * 64l;
  for (int e = threadIdx.x; e < 64 * R; e += 256) {
    if (a) s[e % 64][e / 64] = e / 64 < r ? A[(long)(e / 64) * H + at + e % 64] : f2bf(0.f);
    else s[e / R][e % R] = e % R < r ? B[(at + e / R) * r + e % R] : f2bf(0.f);
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 64 * R; e += 256) {
    if (a) At[at * R + e] = s[e / R][e % R];
    else Bt[(long)(e / 64) * O + at + e % 64] = s[e % 64][e / 64];
  }
}

// Parts of the rows: two workgroups a CU, of 256 rows or more each (a part's sums are 128 bytes a column, and are read
// again).
void split(Outer& a) {
  const long strips = (a.C + STRIP - 1) / STRIP;
  const long parts = std::max(1l, std::min(512 / strips, (long)a.M / 256));
  a.per = (int)(((a.M + parts - 1) / parts + 63) / 64 * 64);
  a.parts = (a.M + a.per - 1) / a.per;
}

template <int R, bool ACROSS>
void outer(const at::Tensor& x, const at::Tensor& y, at::Tensor& out, double scale, hipStream_t stream) {
  Outer a{reinterpret_cast<const bf16*>(x.data_ptr()), reinterpret_cast<const bf16*>(y.data_ptr()),
          reinterpret_cast<bf16*>(out.data_ptr()), nullptr, (int)x.size(0), (int)x.size(1), (int)y.size(1),
          (int)out.size(ACROSS ? 0 : 1), 0, 0, (float)scale};
  split(a);
  at::Tensor part;
  if (a.parts > 1) {
    part = at::empty({a.parts * out.numel()}, x.options().dtype(at::kFloat));
    a.part = part.data_ptr<float>();
  }
  hipLaunchKernelGGL((lora_outer_kernel<R, ACROSS>), dim3((unsigned)((a.C + STRIP - 1) / STRIP * a.parts)), dim3(256),
                     2 * (32768 + R * 128), stream, a);
  HIP_CHECK_KERNEL();
  if (a.parts > 1) {
    hipLaunchKernelGGL(add_outer_kernel, dim3((unsigned)((out.numel() / 4 + 255) / 256)), dim3(256), 0, stream, a.part,
                       a.out, out.numel(), a.parts, a.scale);
    HIP_CHECK_KERNEL();
  }
}

}  // namespace

// g [M, O], x [M, H], A [r, H], B [O, r], tt = (x A^T)^T [R, M rounded up to 64] (lora_forward)
// -> {dA, dB, dt [M, R], A^T [H, R]}
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> lora_grads(const at::Tensor& g, const at::Tensor& x,
                                                                      const at::Tensor& A, const at::Tensor& B,
                                                                      const at::Tensor& tt, double scale) {
  TORCH_CHECK(g.is_cuda() && g.dim() == 2 && x.dim() == 2 && A.dim() == 2 && B.dim() == 2 && tt.dim() == 2,
              "lora_grads: matrices on the GPU");
  const int64_t M = g.size(0), O = g.size(1), H = x.size(1), r = A.size(0), R = r <= 32 ? 32 : 64,
                pitch = (M + 63) / 64 * 64;
  for (const at::Tensor* t : {&g, &x, &A, &B, &tt})
    TORCH_CHECK(t->device() == g.device() && t->scalar_type() == at::kBFloat16 && t->is_contiguous() &&
                    (uintptr_t)t->data_ptr() % 16 == 0, "lora_grads: bf16, whole, at multiples of 16 bytes");
  TORCH_CHECK(x.size(0) == M && A.size(1) == H && B.size(0) == O && B.size(1) == r && tt.size(0) == R &&
                  tt.size(1) == pitch, "lora_grads: shapes");
  TORCH_CHECK(r >= 8 && r <= 64 && r % 8 == 0 && H % 64 == 0 && O % 64 == 0 && M >= 1 && std::max({M, O, H}) < (1l << 23),
              "lora_grads: r a multiple of 8 up to 64, H%64==0, O%64==0, sizes below 2^23");
  const c10::DeviceGuard guard(g.device());
  const auto stream = c10::hip::getCurrentHIPStream().stream();
  auto dA = at::empty_like(A), dB = at::empty_like(B), At = at::empty({H, R}, A.options()),
       Bt = at::empty({R, O}, A.options()), dt = at::empty({M, R}, A.options()), dtt = at::empty({R, pitch}, A.options());
  const auto run = [&](auto rank) {
    constexpr int RANK = rank.value;
    hipLaunchKernelGGL((turn_kernel<RANK>), dim3((unsigned)((H + O) / 64)), dim3(256), 0, stream,
                       reinterpret_cast<const bf16*>(A.data_ptr()), reinterpret_cast<const bf16*>(B.data_ptr()),
                       reinterpret_cast<bf16*>(At.data_ptr()), reinterpret_cast<bf16*>(Bt.data_ptr()), (int)H, (int)O,
                       (int)r);
    HIP_CHECK_KERNEL();
    outer<RANK, false>(g, tt, dB, scale, stream);
    lora_down(g, Bt, r, &dt, &dtt, scale, scale);
    outer<RANK, true>(x, dtt, dA, 1., stream);
  };
  if (R == 32) run(std::integral_constant<int, 32>{});
  else run(std::integral_constant<int, 64>{});
  return {dA, dB, dt, At};
}

}  // namespace amd_ops
