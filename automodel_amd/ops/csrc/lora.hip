// LoRA forward (CDNA4): out = y + scale * (x A^T) B^T in two kernels: the first forms
// t = x A^T (bf16, [M, r]; the backward uses it too), the second adds its product with B to
// the base projection's output in one pass over it.
//
// One kernel per 256 rows did both before, so that 8192 rows were 32 workgroups on 256 CUs
// (600 us on average over the projections of an 8B layer, and a separate addition). Now, at
// 8192 rows: 4096 -> 6144: 70 us, -> 28672: 282, 4096 -> 4096: 48, 14336 -> 4096: 116 (reading x and
// y and writing out at 4.8 TB/s: 56, 210, 42, 77).
//
// Shapes: x [M, H] bf16, A [r, H], B [O, r], r in {32, 64}, H % 64 == 0, O % 64 == 0.
// Below: the segmented kernel for several adapters in one batch (serving).
//
// Reference: nemo_automodel/components/_peft/lora_kernel.py:182 (lora_forward_kernel).

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include "common.h"
#include "ops_api.h"

namespace amd_ops {

typedef __bf16 bf16x8l __attribute__((ext_vector_type(8)));
typedef float f32x4l __attribute__((ext_vector_type(4)));

// [row][64-col] LDS tiles, 128-B rows: same rotation as the grouped kernels
__device__ __forceinline__ int lra_off(int row, int byte_in_row) {
  return row * 128 + (byte_in_row ^ (((row >> 1) & 7) << 4));
}

// t[M, R] = x[M, H] A[R, H]^T. Bound by reading x: 32 rows a workgroup, so that 8192 rows
// fill the chip, and its waves take a quarter of H each, with 4 x 16 bytes of every row in
// flight a lane; A comes from L2. Fragments are loaded straight from memory (a row's 64
// bytes a load; the next load takes the rest of the line from the L1).
template <int R>
__global__ __launch_bounds__(256) void lora_down_kernel(const bf16* __restrict__ x,
                                                        const bf16* __restrict__ A,
                                                        bf16* __restrict__ t, long M, int H) {
  constexpr int U = 4;
  __shared__ float red[4][32][R + 1];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, l16 = lane & 15, kq = lane >> 4;
  const long m0 = (long)blockIdx.x * 32;
  const bf16* xr[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) xr[i] = x + min(m0 + i * 16 + l16, M - 1) * H + kq * 8;
  const bf16* ar = A + (long)l16 * H + kq * 8;
  f32x4l acc[2][R / 16];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < R / 16; ++j) acc[i][j] = f32x4l{0.f, 0.f, 0.f, 0.f};
  const int per = (H / 32 + 3) / 4 * 32;               // H is a multiple of 64
  const int k1 = min((wid + 1) * per, H);
  for (int k = wid * per; k < k1; k += 32 * U) {
    bf16x8l xv[U][2], av[U][R / 16];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kk = min(k + 32 * u, k1 - 32);         // (beyond the end: loaded, not added)
#pragma unroll
      for (int i = 0; i < 2; ++i) xv[u][i] = *reinterpret_cast<const bf16x8l*>(xr[i] + kk);
#pragma unroll
      for (int j = 0; j < R / 16; ++j)
        av[u][j] = *reinterpret_cast<const bf16x8l*>(ar + (long)j * 16 * H + kk);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k + 32 * u < k1) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < R / 16; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xv[u][i], av[u][j], acc[i][j], 0, 0, 0);
      }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < R / 16; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[wid][i * 16 + kq * 4 + v][j * 16 + l16] = acc[i][j][v];
  __syncthreads();
  for (int e = threadIdx.x; e < 32 * R; e += 256) {
    const int m = e / R, r = e % R;
    if (m0 + m < M)
      t[(m0 + m) * R + r] = f2bf(red[0][m][r] + red[1][m][r] + red[2][m][r] + red[3][m][r]);
  }
}

// out[M, O] = y + scale * t[M, R] B[O, R]^T (without y: the product alone). Bound by y and
// out. A wave takes 16 rows x 64 columns a step: the rows of B lie in the MFMAs in an order
// that leaves a lane 16 consecutive columns of one row.
template <int R>
__global__ __launch_bounds__(256) void lora_up_kernel(const bf16* __restrict__ y,
                                                      const bf16* __restrict__ t,
                                                      const bf16* __restrict__ B,
                                                      bf16* __restrict__ out, long M, int O,
                                                      float scale) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, l16 = lane & 15, g = lane >> 4;
  const int strips = (O + 255) / 256;                  // blocks side by side take one stretch of rows
  const long m = (long)(blockIdx.x / strips) * 64 + wid * 16 + l16;
  const bf16* tr = t + min(m, M - 1) * R + g * 8;
  bf16x8l tv[R / 32];
#pragma unroll
  for (int kk = 0; kk < R / 32; ++kk) tv[kk] = *reinterpret_cast<const bf16x8l*>(tr + kk * 32);
  const int perm = (l16 >> 2) * 16 + (l16 & 3);        // column of row l16 of tile j: perm + 4 j
#pragma unroll 2
  for (int s = 0; s < 4; ++s) {
    const int o0 = blockIdx.x % strips * 256 + s * 64;
    if (o0 >= O) break;                                // O is a multiple of 64
    const long at = m * O + o0 + g * 16;
    bf16x8 yv[2];
    if (y && m < M) {
      yv[0] = *reinterpret_cast<const bf16x8*>(y + at);
      yv[1] = *reinterpret_cast<const bf16x8*>(y + at + 8);
    }
    f32x4l acc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc[j] = f32x4l{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < R / 32; ++kk) {
        const bf16x8l b = *reinterpret_cast<const bf16x8l*>(
            B + (long)(o0 + perm + j * 4) * R + kk * 32 + g * 8);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, tv[kk], acc[j], 0, 0, 0);
      }
    }
    if (m < M) {
      bf16x8 w[2];
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float d = acc[e >> 2][e & 3] * scale;
        w[e >> 3].v[e & 7] = f2bf(y ? bf2f(yv[e >> 3].v[e & 7]) + d : d);
      }
      *reinterpret_cast<bf16x8*>(out + at) = w[0];
      *reinterpret_cast<bf16x8*>(out + at + 8) = w[1];
    }
  }
}

// ===========================================================================
// SGMV: segmented multi-adapter fused LoRA (serving path — SURVEY §2.9
// "SGMV kernels"; reference uses punica-style segmented gather MV for
// per-request adapters). Tokens arrive SORTED by adapter; the grouped-GEMM
// plan (offs + 256-row tile_map, device-built) picks each tile's adapter,
// whose A/B/scale are indexed from stacked tensors. One kernel per 256 rows
// does both products: the first one's result goes through LDS as the second's
// operand.
// ===========================================================================

template <int R>
__global__ __launch_bounds__(256) void sgmv_fused_fwd_kernel(
    const bf16* __restrict__ x, const bf16* __restrict__ A, const bf16* __restrict__ B,
    const float* __restrict__ scales, bf16* __restrict__ out,
    const int* __restrict__ tile_map, const int* __restrict__ offs,
    const int* __restrict__ n_tiles, int H, int O) {
  if (n_tiles != nullptr && (int)blockIdx.x >= n_tiles[0]) return;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* a_lds = smem;
  char* t_lds = smem + R * 128;
  char* b_lds = t_lds + 256 * R * 2;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = tid >> 6;
  const int l16 = lane & 15;
  const int kq = lane >> 4;

  const int ad = tile_map[2 * blockIdx.x];
  const long m0 = tile_map[2 * blockIdx.x + 1];
  const long m_end = offs[ad + 1];
  const float scale = scales[ad];
  const bf16* Aa = A + (long)ad * R * H;
  const bf16* Ba = B + (long)ad * O * R;
  const int mw = wid * 64;

  f32x4l acc1[4][R / 16];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < R / 16; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc1[i][j][v] = 0.f;

  for (int h0 = 0; h0 < H; h0 += 64) {
    for (int idx = tid; idx < R * 8; idx += 256) {
      const int r = idx / 8, c = (idx % 8) * 8;
      *reinterpret_cast<bf16x8*>(a_lds + lra_off(r, c * 2)) =
          *reinterpret_cast<const bf16x8*>(Aa + (long)r * H + h0 + c);
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8l b[R / 16];
#pragma unroll
      for (int j = 0; j < R / 16; ++j)
        b[j] = *reinterpret_cast<const bf16x8l*>(
            a_lds + lra_off(j * 16 + l16, (kk * 32 + kq * 8) * 2));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const long m = m0 + mw + i * 16 + l16;
        bf16x8l a;
        if (m < m_end) {
          a = *reinterpret_cast<const bf16x8l*>(x + m * H + h0 + kk * 32 + kq * 8);
        } else {
#pragma unroll
          for (int v = 0; v < 8; ++v) a[v] = (__bf16)0.f;
        }
#pragma unroll
        for (int j = 0; j < R / 16; ++j)
          acc1[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[j], acc1[i][j], 0, 0, 0);
      }
    }
    __syncthreads();
  }

  {
    char* tw = t_lds + (long)(mw) * R * 2;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < R / 16; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int m = i * 16 + kq * 4 + v;
          const int r = j * 16 + l16;
          *reinterpret_cast<bf16*>(tw + (long)m * R * 2 + r * 2) =
              f2bf(acc1[i][j][v]);
        }
  }
  __syncthreads();

  for (int o0 = 0; o0 < O; o0 += 64) {
    for (int idx = tid; idx < 64 * (R / 8); idx += 256) {
      const int o = idx / (R / 8), c = (idx % (R / 8)) * 8;
      *reinterpret_cast<bf16x8*>(b_lds + lra_off(o, c * 2)) =
          *reinterpret_cast<const bf16x8*>(Ba + (long)(o0 + o) * R + c);
    }
    __syncthreads();

    f32x4l acc2[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc2[i][j][v] = 0.f;

    const char* tw = t_lds + (long)(mw) * R * 2;
#pragma unroll
    for (int kk = 0; kk < R / 32; ++kk) {
      bf16x8l bfr[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        bfr[j] = *reinterpret_cast<const bf16x8l*>(
            b_lds + lra_off(j * 16 + l16, (kk * 32 + kq * 8) * 2));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bf16x8l a = *reinterpret_cast<const bf16x8l*>(
            tw + (long)(i * 16 + l16) * R * 2 + (kk * 32 + kq * 8) * 2);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc2[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bfr[j], acc2[i][j], 0, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const long m = m0 + mw + i * 16 + kq * 4 + v;
        if (m < m_end) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            out[m * O + o0 + j * 16 + l16] = f2bf(acc2[i][j][v] * scale);
        }
      }
    }
    __syncthreads();
  }
}

at::Tensor sgmv_fused_fwd(const at::Tensor& x, const at::Tensor& A, const at::Tensor& B,
                          const at::Tensor& scales, const at::Tensor& offs,
                          const at::Tensor& tile_map,
                          const std::optional<at::Tensor>& n_tiles) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.scalar_type() == at::kBFloat16,
              "sgmv_fused_fwd: x [M,H] bf16");
  TORCH_CHECK(A.dim() == 3 && B.dim() == 3, "A [n,r,H], B [n,O,r]");
  const long M = x.size(0);
  const int H = x.size(1), R = A.size(1), O = B.size(1);
  TORCH_CHECK(A.size(2) == H && B.size(2) == R && A.size(0) == B.size(0),
              "shape mismatch");
  TORCH_CHECK((R == 32 || R == 64) && H % 64 == 0 && O % 64 == 0,
              "sgmv: r in {32, 64}, H%64==0, O%64==0");
  TORCH_CHECK(scales.scalar_type() == at::kFloat && scales.numel() == A.size(0),
              "scales: float32 [n_adapters]");
  auto out = at::empty({M, (long)O}, x.options());
  const int nt = tile_map.size(0);
  if (M == 0 || nt == 0) return out;
  const size_t smem = R * 128 + 256 * R * 2 + 64 * 128;
  auto stream = c10::hip::getCurrentHIPStream();
  const int* ntp = n_tiles.has_value() ? n_tiles->data_ptr<int>() : nullptr;
  if (R == 32) {
    hipLaunchKernelGGL((sgmv_fused_fwd_kernel<32>), dim3(nt), dim3(256), smem,
                       stream.stream(),
                       reinterpret_cast<const bf16*>(x.data_ptr()),
                       reinterpret_cast<const bf16*>(A.data_ptr()),
                       reinterpret_cast<const bf16*>(B.data_ptr()),
                       scales.data_ptr<float>(),
                       reinterpret_cast<bf16*>(out.data_ptr()),
                       tile_map.data_ptr<int>(), offs.data_ptr<int>(), ntp, H, O);
  } else {
    hipLaunchKernelGGL((sgmv_fused_fwd_kernel<64>), dim3(nt), dim3(256), smem,
                       stream.stream(),
                       reinterpret_cast<const bf16*>(x.data_ptr()),
                       reinterpret_cast<const bf16*>(A.data_ptr()),
                       reinterpret_cast<const bf16*>(B.data_ptr()),
                       scales.data_ptr<float>(),
                       reinterpret_cast<bf16*>(out.data_ptr()),
                       tile_map.data_ptr<int>(), offs.data_ptr<int>(), ntp, H, O);
  }
  HIP_CHECK_KERNEL();
  return out;
}

// -> (y + scale * (x A^T) B^T, x A^T)
std::tuple<at::Tensor, at::Tensor> lora_apply(const std::optional<at::Tensor>& y, const at::Tensor& x,
                                              const at::Tensor& A, const at::Tensor& B, double scale) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.scalar_type() == at::kBFloat16 && x.is_contiguous(),
              "lora_apply: x [M,H] bf16");
  const long M = x.size(0);
  const int H = x.size(1), R = A.size(0), O = B.size(0);
  TORCH_CHECK(A.dim() == 2 && B.dim() == 2 && A.size(1) == H && B.size(1) == R, "shape mismatch");
  TORCH_CHECK(A.scalar_type() == at::kBFloat16 && B.scalar_type() == at::kBFloat16 && A.is_contiguous() &&
                  B.is_contiguous(), "lora_apply: A [r,H], B [O,r] bf16");
  TORCH_CHECK((R == 32 || R == 64) && H % 64 == 0 && O % 64 == 0,
              "lora: r in {32, 64}, H%64==0, O%64==0");
  if (y)
    TORCH_CHECK(y->is_cuda() && y->dim() == 2 && y->size(0) == M && y->size(1) == O && y->is_contiguous() &&
                    y->scalar_type() == at::kBFloat16, "lora_apply: y [M,O] bf16");
  auto out = at::empty({M, (long)O}, x.options());
  auto t = at::empty({M, (long)R}, x.options());
  if (M == 0) return {out, t};
  const long blocks = (M + 63) / 64 * ((O + 255) / 256);
  // (a grid has 2^32 threads)
  TORCH_CHECK(blocks < (1l << 24) && (M + 31) / 32 < (1l << 24), "lora_apply: too many rows");
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const bf16* yp = y ? reinterpret_cast<const bf16*>(y->data_ptr()) : nullptr;
  auto run = [&](auto rank) {
    constexpr int RANK = rank.value;
    hipLaunchKernelGGL((lora_down_kernel<RANK>), dim3((unsigned)((M + 31) / 32)), dim3(256), 0, stream,
                       reinterpret_cast<const bf16*>(x.data_ptr()),
                       reinterpret_cast<const bf16*>(A.data_ptr()),
                       reinterpret_cast<bf16*>(t.data_ptr()), M, H);
    hipLaunchKernelGGL((lora_up_kernel<RANK>), dim3((unsigned)blocks), dim3(256), 0, stream, yp,
                       reinterpret_cast<const bf16*>(t.data_ptr()),
                       reinterpret_cast<const bf16*>(B.data_ptr()),
                       reinterpret_cast<bf16*>(out.data_ptr()), M, O, (float)scale);
  };
  if (R == 32) run(std::integral_constant<int, 32>{});
  else run(std::integral_constant<int, 64>{});
  HIP_CHECK_KERNEL();
  return {out, t};
}

at::Tensor lora_fused_fwd(const at::Tensor& x, const at::Tensor& A, const at::Tensor& B,
                          double scale) {
  return std::get<0>(lora_apply(std::nullopt, x.contiguous(), A.contiguous(), B.contiguous(), scale));
}

}  // namespace amd_ops
