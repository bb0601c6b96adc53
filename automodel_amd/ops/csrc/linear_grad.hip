// Gradients of y = x w^T in bf16 with f32 accumulation (gfx950), by the tiles of gemm_tile.h:
//
//   linear_dw   dw[n, k] = sum_t g[t, n] x[t, k]
//   linear_dx   dx[t, k] = sum_n g[t, n] w[n, k]
//
// Both take their operands as they are.
#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include "common.h"
#include "gemm_tile.h"
#include "ops_api.h"

namespace amd_ops {

namespace {

struct Args {
  const bf16 *r, *c;
  bf16* out;
  int rows, cols, sum;
};

// Blocks are dealt to the 8 XCDs in contiguous stretches of the tile list, whose order is
// down 4 row tiles, then on to the next column tile: the 32 tiles of an XCD at a time read
// 4 row tiles and 8 column tiles.
constexpr int DOWN = 4;

template <bool DW>
__global__ __launch_bounds__(gt::THREADS, 1) void linear_grad_kernel(const Args a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int nr = (a.rows + gt::TILE - 1) / gt::TILE, nc = (a.cols + gt::TILE - 1) / gt::TILE;
  const int total = nr * nc, per = (total + 7) / 8, slot = blockIdx.x >> 3, id = (blockIdx.x & 7) * per + slot;
  if (slot >= per || id >= total) return;
  const int group = id / (DOWN * nc), in = id % (DOWN * nc), down = min(DOWN, nr - group * DOWN);
  const int r0 = (group * DOWN + in % down) * gt::TILE, c0 = in / down * gt::TILE;
  gt::Tile t{};
  t.rows = a.rows - r0;
  t.cols = a.cols - c0;
  t.sum = t.after = a.sum;
  t.r_ld = DW ? a.rows : a.sum;
  t.c_ld = a.cols;
  t.r = DW ? a.r + r0 : a.r + (long)r0 * a.sum;
  t.c = a.c + c0;
  gt::f32x4_t acc[8][8];
  gt::multiply<DW>(acc, t, smem);
  gt::store(acc, smem, a.out + (long)r0 * a.cols + c0, a.cols, t.rows, t.cols);
}

template <bool DW>
at::Tensor run(const at::Tensor& r, const at::Tensor& c, int64_t rows, int64_t cols, int64_t sum) {
  TORCH_CHECK(r.is_cuda() && r.device() == c.device() && r.is_contiguous() && c.is_contiguous() &&
                  r.scalar_type() == at::kBFloat16 && c.scalar_type() == at::kBFloat16,
              "linear_grad: contiguous bf16 operands on one GPU");
  TORCH_CHECK((uintptr_t)r.data_ptr() % 16 == 0 && (uintptr_t)c.data_ptr() % 16 == 0,
              "linear_grad: operands at multiples of 16 bytes");
  // a tile's addresses are 32 bits: 256 rows of 2^23
  TORCH_CHECK(std::max({rows, cols, sum}) < (1l << 23), "linear_grad: sizes below 2^23");
  const c10::DeviceGuard guard(r.device());
  auto out = at::empty({rows, cols}, r.options());
  if (out.numel() == 0) return out;
  const Args a{reinterpret_cast<const bf16*>(r.data_ptr()), reinterpret_cast<const bf16*>(c.data_ptr()),
               reinterpret_cast<bf16*>(out.data_ptr()), (int)rows, (int)cols, (int)sum};
  const long tiles = ((rows + gt::TILE - 1) / gt::TILE) * ((cols + gt::TILE - 1) / gt::TILE);
  // the stretches of the 8 XCDs are rounded up: up to 7 workgroups beyond the tiles
  hipLaunchKernelGGL((linear_grad_kernel<DW>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(gt::THREADS),
                     gt::SMEM, c10::hip::getCurrentHIPStream().stream(), a);
  HIP_CHECK_KERNEL();
  return out;
}

}  // namespace

at::Tensor linear_dw(const at::Tensor& g, const at::Tensor& x) {
  TORCH_CHECK(g.dim() == 2 && x.dim() == 2 && g.size(0) == x.size(0), "linear_dw: g [T, N], x [T, K]");
  TORCH_CHECK(g.size(0) > 0 && g.size(1) % 8 == 0 && x.size(1) % 8 == 0, "linear_dw: rows, N%8 == 0, K%8 == 0");
  return run<true>(g, x, g.size(1), x.size(1), g.size(0));
}

at::Tensor linear_dx(const at::Tensor& g, const at::Tensor& w) {
  TORCH_CHECK(g.dim() == 2 && w.dim() == 2 && g.size(1) == w.size(0), "linear_dx: g [T, N], w [N, K]");
  TORCH_CHECK(w.size(0) > 0 && w.size(0) % (2 * gt::STEP) == 0 && w.size(1) % 8 == 0,
              "linear_dx: N%64 == 0, K%8 == 0");
  return run<false>(g, w, g.size(0), w.size(1), w.size(0));
}

}  // namespace amd_ops
