// LoRA forward (CDNA4): out = y + scale * (x A^T) B^T in two kernels: the first forms
// t = x A^T (bf16, [M, r]; the backward uses it too), the second adds its product with B to
// the base projection's output in one pass over it.
//
// One kernel per 256 rows did both before, so that 8192 rows were 32 workgroups on 256 CUs
// (600 us on average over the projections of an 8B layer, and a separate addition). Now, at
// 8192 rows: 4096 -> 6144: 60 us, -> 28672: 272, 4096 -> 4096: 38, 14336 -> 4096: 88 (reading x and
// y and writing out at 4.8 TB/s: 56, 210, 42, 77).
//
// Where the base layer is a plain frozen one in training, its own tiles have the second product behind their sums instead
// (linear_grad.hip: lora_linear), and only t is formed here.
//
// Shapes: x [M, H] bf16, A [r, H], B [O, r], H % 64 == 0, O % 64 == 0; r 32 or 64, or a multiple of 8 below,
// which the kernels fill up with zeros.
// Below: the segmented kernel for several adapters in one batch (serving).
//
// Reference: nemo_automodel/components/_peft/lora_kernel.py:182 (lora_forward_kernel).

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include "common.h"
#include "gemm_tile.h"
#include "ops_api.h"

namespace amd_ops {

typedef __bf16 bf16x8l __attribute__((ext_vector_type(8)));
typedef float f32x4l __attribute__((ext_vector_type(4)));

// [row][64-col] LDS tiles, 128-B rows: same rotation as the grouped kernels
__device__ __forceinline__ int lra_off(int row, int byte_in_row) {
  return row * 128 + (byte_in_row ^ (((row >> 1) & 7) << 4));
}

struct Down {
  const bf16 *x, *A;
  bf16 *t, *turned;          // turned: or null
  long M, pitch;
  int H, r;                  // r: rows of A, R at most; columns of t behind them are zeros, whatever x is
  float scale, scale_turned;
};

constexpr int DOWN = 32;     // rows of a workgroup

// t[M, R] = scale x[M, H] A[R, H]^T, and, where they are wanted, its columns as rows of M rounded up to 64
// (`pitch`), zeros behind M, by a scale of their own. Bound by reading x: 32 rows a workgroup, so that 8192 rows fill the chip, and its waves
// take a quarter of H each, 64 columns a step: their own stretches of x and of A (from the L2) come straight to
// their own LDS, three steps ahead (R 64: two), with no barrier in the loop. 8192 x 28672 90 us, 8192 x 4096 14.
// (Fragments straight from memory, four of each in flight: 158, 3.0 TB/s, and 23.)
template <int R>
__global__ __launch_bounds__(256, 1) void lora_down_kernel(const Down a) {
  constexpr int LOADS = DOWN / 8 + R / 8, SLOT = LOADS * 1024, SLOTS = R == 32 ? 4 : 3;
  extern __shared__ __attribute__((aligned(1024))) char down_smem[];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const long m0 = (long)blockIdx.x * DOWN;
  const int per = (a.H / 32 + 3) / 4 * 32;             // H is a multiple of 64
  const int k0 = min(wid * per, a.H), left = min((wid + 1) * per, a.H) - k0, n = (left + 63) / 64;
  const unsigned ld = 2u * a.H;
  // 8 rows of 64 columns a load; pieces of 16 bytes permuted by row for the rows that meet in a read
  unsigned off[R / 8];
#pragma unroll
  for (int h = 0; h < R / 8; ++h) off[h] = (8 * h + (lane >> 3)) * ld + ((lane & 7) ^ ((4 * h + (lane >> 4)) & 7)) * 16;
  const int have = (int)max(0l, min(a.M - m0, (long)DOWN));
  const char *xp = reinterpret_cast<const char*>(a.x + (have ? m0 * a.H + k0 : 0));
  const char* ap = reinterpret_cast<const char*>(a.A + k0);
  // bytes to the tensors' ends; none of what is behind the wave's columns
  unsigned xn = have ? have * ld - 2 * k0 : 0, an = a.r * ld - 2 * k0;
  int ahead = n;
  const unsigned mine = fa::lds_address(down_smem) + wid * (SLOTS * SLOT);
  auto load = [&](unsigned to) __attribute__((always_inline)) {
    const unsigned x_end = ahead > 0 ? xn : 0, a_end = ahead > 0 ? an : 0;
#pragma unroll
    for (int h = 0; h < DOWN / 8; ++h) gt::load_lds(to, h * 1024, off[h], xp, x_end);
#pragma unroll
    for (int h = 0; h < R / 8; ++h) gt::load_lds(to, DOWN * 128 + h * 1024, off[h], ap, a_end);
    xp += 128;
    ap += 128;
    xn -= 128;
    an -= 128;
    ahead -= 1;
  };
  f32x4l acc[2][R / 16];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < R / 16; ++j) acc[i][j] = f32x4l{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < SLOTS; ++p) load(mine + p * SLOT);
  unsigned slot = mine;
#pragma unroll 1
  for (int p = 0; p < n; ++p) {
    fa::wait_loads<(SLOTS - 1) * LOADS>();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      if (p * 64 + q * 32 >= left) break;              // (the quarters are multiples of 32)
      typedef __attribute__((address_space(3))) bf16x8l* lds_ptr;
      const unsigned at = slot + l16 * 128 + (((q * 4 + g) ^ (l16 >> 1)) << 4);
      bf16x8l xv[2], av[R / 16];
#pragma unroll
      for (int i = 0; i < 2; ++i) xv[i] = *(lds_ptr)(uintptr_t)(at + i * 2048);
#pragma unroll
      for (int j = 0; j < R / 16; ++j) av[j] = *(lds_ptr)(uintptr_t)(at + DOWN * 128 + j * 2048);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < R / 16; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xv[i], av[j], acc[i][j], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    load(slot);
    slot = slot == mine + (SLOTS - 1) * SLOT ? mine : slot + SLOT;
  }
  fa::wait_loads();
  fa::barrier();
  float(*red)[DOWN][R + 1] = reinterpret_cast<float(*)[DOWN][R + 1]>(down_smem);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < R / 16; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[wid][i * 16 + g * 4 + v][j * 16 + l16] = acc[i][j][v];
  __syncthreads();
  auto sum = [&](int m, int r, float scale) {          // (0 x infinity is none)
    return r < a.r ? (red[0][m][r] + red[1][m][r] + red[2][m][r] + red[3][m][r]) * scale : 0.f;
  };
  for (int e = threadIdx.x; e < DOWN * R; e += 256)
    if (e / R < have) a.t[m0 * R + e] = f2bf(sum(e / R, e % R, a.scale));
  if (!a.turned) return;
  for (int e = threadIdx.x; e < DOWN * R; e += 256)
    a.turned[e / DOWN * a.pitch + m0 + e % DOWN] = f2bf(e % DOWN < have ? sum(e % DOWN, e / DOWN, a.scale_turned) : 0.f);
}

// out[M, O] = y + scale * t[M, R] B[O, R]^T (without y: the product alone). Bound by y and
// out. A wave takes 16 rows x 64 columns a step: the rows of B lie in the MFMAs in an order
// that leaves a lane 16 consecutive columns of one row.
template <int R>
__global__ __launch_bounds__(256) void lora_up_kernel(const bf16* __restrict__ y,
                                                      const bf16* __restrict__ t,
                                                      const bf16* __restrict__ B,
                                                      bf16* __restrict__ out, long M, int O, int r,
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
        bf16x8l b = {};                                // r is a multiple of 8
        if (kk * 32 + g * 8 < r)
          b = *reinterpret_cast<const bf16x8l*>(B + (long)(o0 + perm + j * 4) * r + kk * 32 + g * 8);
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

// t = scale x A^T [M, r rounded up to 32] of A's first r rows, with zeros behind r, and scale_turned (x A^T)^T, M rounded up
// to 64, with zeros behind M; x and A at multiples of 16 bytes
void lora_down(const at::Tensor& x, const at::Tensor& A, int64_t r, at::Tensor* t, at::Tensor* turned, double scale,
               double scale_turned) {
  const long M = x.size(0), pitch = (M + 63) / 64 * 64, blocks = ((turned ? pitch : M) + DOWN - 1) / DOWN;
  // (a grid has 2^32 threads; a lane's offsets of 64 rows are 32 bits)
  TORCH_CHECK(blocks < 1l << 24 && x.size(1) < 1l << 25, "lora: too many rows or columns");
  const Down a{reinterpret_cast<const bf16*>(x.data_ptr()), reinterpret_cast<const bf16*>(A.data_ptr()),
               reinterpret_cast<bf16*>(t->data_ptr()), turned ? reinterpret_cast<bf16*>(turned->data_ptr()) : nullptr, M,
               pitch, (int)x.size(1), (int)r, (float)scale, (float)scale_turned};
  const auto launch = [&](auto rank) {
    constexpr int RANK = rank.value, smem = 4 * (RANK == 32 ? 4 : 3) * (DOWN / 8 + RANK / 8) * 1024;
    hipLaunchKernelGGL((lora_down_kernel<RANK>), dim3((unsigned)blocks), dim3(256), smem,
                       c10::hip::getCurrentHIPStream().stream(), a);
  };
  if (t->size(1) == 32) launch(std::integral_constant<int, 32>{});
  else launch(std::integral_constant<int, 64>{});
  HIP_CHECK_KERNEL();
}

namespace {

// -> (y + scale * (x A^T) B^T, x A^T, (x A^T)^T if it is wanted)
std::tuple<at::Tensor, at::Tensor, at::Tensor> forward(const std::optional<at::Tensor>& y, const at::Tensor& x,
                                                       const at::Tensor& A, const at::Tensor& B, double scale,
                                                       bool turn) {
  TORCH_CHECK(x.is_cuda() && x.dim() == 2 && x.scalar_type() == at::kBFloat16 && x.is_contiguous(),
              "lora_apply: x [M,H] bf16");
  const long M = x.size(0);
  const int H = x.size(1), r = A.size(0), R = r <= 32 ? 32 : 64, O = B.size(0);
  TORCH_CHECK(A.dim() == 2 && B.dim() == 2 && A.size(1) == H && B.size(1) == r, "shape mismatch");
  TORCH_CHECK(A.scalar_type() == at::kBFloat16 && B.scalar_type() == at::kBFloat16 && A.is_contiguous() &&
                  B.is_contiguous(), "lora_apply: A [r,H], B [O,r] bf16");
  TORCH_CHECK(r >= 8 && r <= 64 && r % 8 == 0 && H % 64 == 0 && O % 64 == 0,
              "lora: r a multiple of 8 up to 64, H%64==0, O%64==0");
  if (y)
    TORCH_CHECK(y->is_cuda() && y->dim() == 2 && y->size(0) == M && y->size(1) == O && y->is_contiguous() &&
                    y->scalar_type() == at::kBFloat16, "lora_apply: y [M,O] bf16");
  auto out = at::empty({M, (long)O}, x.options());
  auto t = at::empty({M, (long)R}, x.options());
  at::Tensor turned;
  if (turn) turned = at::empty({R, (M + 63) / 64 * 64}, x.options());
  if (M == 0) return {out, t, turned};
  const long blocks = (M + 63) / 64 * ((O + 255) / 256);
  // (a grid has 2^32 threads)
  TORCH_CHECK(blocks < (1l << 24), "lora_apply: too many rows");
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const bf16* yp = y ? reinterpret_cast<const bf16*>(y->data_ptr()) : nullptr;
  // lora_down's loads take whole pieces of 16 bytes; a view into a larger buffer may lie anywhere
  const auto whole = [](const at::Tensor& v) { return (uintptr_t)v.data_ptr() % 16 ? v.clone() : v; };
  auto run = [&](auto rank) {
    constexpr int RANK = rank.value;
    lora_down(whole(x), whole(A), r, &t, turn ? &turned : nullptr, 1., 1.);
    hipLaunchKernelGGL((lora_up_kernel<RANK>), dim3((unsigned)blocks), dim3(256), 0, stream, yp,
                       reinterpret_cast<const bf16*>(t.data_ptr()),
                       reinterpret_cast<const bf16*>(B.data_ptr()),
                       reinterpret_cast<bf16*>(out.data_ptr()), M, O, r, (float)scale);
  };
  if (R == 32) run(std::integral_constant<int, 32>{});
  else run(std::integral_constant<int, 64>{});
  HIP_CHECK_KERNEL();
  return {out, t, turned};
}

}  // namespace

// r a multiple of 8 up to 64 -> (y + scale * (x A^T) B^T, x A^T [M, r rounded up to 32] with zeros behind r)
std::tuple<at::Tensor, at::Tensor> lora_apply(const std::optional<at::Tensor>& y, const at::Tensor& x,
                                              const at::Tensor& A, const at::Tensor& B, double scale) {
  const auto r = forward(y, x, A, B, scale, false);
  return {std::get<0>(r), std::get<1>(r)};
}

// -> (the same, (x A^T)^T [r rounded up to 32, M to 64] with zeros behind r and M, which lora_grads reads)
std::tuple<at::Tensor, at::Tensor> lora_forward(const at::Tensor& y, const at::Tensor& x, const at::Tensor& A,
                                                const at::Tensor& B, double scale) {
  const auto r = forward(y, x, A, B, scale, true);
  return {std::get<0>(r), std::get<2>(r)};
}

at::Tensor lora_fused_fwd(const at::Tensor& x, const at::Tensor& A, const at::Tensor& B,
                          double scale) {
  TORCH_CHECK(A.dim() == 2 && (A.size(0) == 32 || A.size(0) == 64), "lora_fused_fwd: r in {32, 64}");
  return std::get<0>(lora_apply(std::nullopt, x.contiguous(), A.contiguous(), B.contiguous(), scale));
}

}  // namespace amd_ops
