// y = x w^T and its gradients in bf16 with f32 accumulation (gfx950), by the tiles of gemm_tile.h:
//
//   linear_y    y[t, n]  = sum_k x[t, k] w[n, k]
//   linear_dw   dw[n, k] = sum_t g[t, n] x[t, k]
//   linear_dx   dx[t, k] = sum_n g[t, n] w[n, k]
//
// All take their operands as they are.
//
// The chip has 256 workgroups, and most layers have not so many tiles of 256 x 256, or a few more (2048 x 2048:
// 64; 6144 x 4096: 384). So tiles have 128 to 256 rows, and a sum can be cut into parts, each a tile of its own
// in 32 bits, which `add_parts_kernel` adds up in their order: what takes least by `predicted`. Against 256
// rows and whole sums, us: dw of 8192 tokens, 2048 x 2048 141 -> 70 (128 rows, 2 parts), 2816 x 2048 141 -> 95
// (256 rows, 2 parts), 6144 x 4096 317 -> 289 (192 rows); dx of 1001 tokens, 6144 x 1536 104 -> 30 (128 rows, 4
// parts). The library: 86, 127, 343, 56. (x w^T has measurements of its own in linear_out.hip.)
#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include "common.h"
#include "linear_tiles.h"
#include "ops_api.h"

namespace amd_ops {

using lg::Args;
using lg::cut;

namespace {

// The parts' sum in bf16. A workgroup has 16 rows of a wave's part of a tile, a thread two pieces of 4 columns: whole
// kilobytes of each part, read once. 33 MB of two parts of 2048 x 2048: 9 us with the launch.
__global__ __launch_bounds__(256) void add_parts_kernel(const Args a) {
  const int nc = (a.cols + gt::TILE - 1) / gt::TILE, nr = (a.rows + a.height - 1) / a.height;
  const int most = a.height / 32, i = blockIdx.x % most, w = blockIdx.x / most % 4, tile = blockIdx.x / most / 4;
  int r0, c0;
  lg::place(tile, nr, nc, a.height, r0, c0);
  const int rows = min(a.rows - r0, a.height), each = gt::rows16(rows);
  if (i >= each) return;
  const int lane = threadIdx.x & 63;
  const long part = (long)nr * nc * a.height * gt::TILE;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int j = (threadIdx.x >> 6) * 2 + q;
    const float* p = a.part + (long)tile * a.height * gt::TILE + ((w * each + i) * 8 + j) * 256 + lane * 4;
    gt::f32x4_t s = *reinterpret_cast<const gt::f32x4_t*>(p);
    for (int k = 1; k < a.parts; ++k) s += *reinterpret_cast<const gt::f32x4_t*>(p + k * part);
    const int row = ((w >> 1) * each + i) * 16 + (lane & 15), col = c0 + (w & 1) * 128 + j * 16 + (lane >> 4) * 4;
    if (row >= rows || col >= a.cols) continue;
    fa::bf16x4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (__bf16)(a.relu2 ? gt::relu2(s[e]) : s[e]);
    *reinterpret_cast<fa::bf16x4_t*>(a.out + (long)(r0 + row) * a.cols + col) = o;
  }
}

template <lg::Form FORM>
at::Tensor run(const at::Tensor& r, const at::Tensor& c, int64_t rows, int64_t cols, int64_t sum,
               const at::Tensor* r2 = nullptr, const at::Tensor* c2 = nullptr, bool relu2 = false, const at::Tensor* up = nullptr) {
  TORCH_CHECK(r.is_cuda() && r.device() == c.device() && r.is_contiguous() && c.is_contiguous() &&
                  r.scalar_type() == at::kBFloat16 && c.scalar_type() == at::kBFloat16,
              "linear_grad: contiguous bf16 operands on one GPU");
  TORCH_CHECK((uintptr_t)r.data_ptr() % 16 == 0 && (uintptr_t)c.data_ptr() % 16 == 0,
              "linear_grad: operands at multiples of 16 bytes");
  // a tile's addresses are 32 bits: 256 rows of 2^23
  TORCH_CHECK(std::max({rows, cols, sum}) < (1l << 23), "linear_grad: sizes below 2^23");
  const c10::DeviceGuard guard(r.device());
  auto out = at::empty({rows, FORM == lg::GLU ? cols / 2 : cols}, r.options());
  if (out.numel() == 0) return out;
  Args a{reinterpret_cast<const bf16*>(r.data_ptr()), reinterpret_cast<const bf16*>(c.data_ptr()),
         reinterpret_cast<bf16*>(out.data_ptr()), nullptr, (int)rows, (int)cols, (int)sum, 0, 0, 0, nullptr, nullptr, 0, 0, relu2,
         up ? reinterpret_cast<const bf16*>(up->data_ptr()) : nullptr};
  if (r2) {
    a.r2 = reinterpret_cast<const bf16*>(r2->data_ptr());
    a.c2 = reinterpret_cast<const bf16*>(c2->data_ptr());
    a.rank = (int)r2->size(1);
    a.rank_c = (int)c2->size(1);
  }
  cut(FORM, a);
  const long tiles = lg::tiles_of(a);
  TORCH_CHECK(tiles * 32 < (1l << 31), "linear_grad: too many tiles");
  at::Tensor part;
  if (a.parts > 1) {
    part = at::empty({a.parts * tiles * a.height * gt::TILE}, r.options().dtype(at::kFloat));
    a.part = part.data_ptr<float>();
  }
  // a workgroup a CU, and no more than tiles, rounded up to the XCDs' equal parts
  const long blocks = std::min((tiles * a.parts + 7) / 8 * 8, gt::workgroups());
  const auto stream = c10::hip::getCurrentHIPStream().stream();
  const auto launch = [&](auto short_, auto parts_) {
    hipLaunchKernelGGL((lg::linear_tile_kernel<FORM, decltype(short_)::value, decltype(parts_)::value>), dim3((unsigned)blocks),
                       dim3(gt::THREADS), gt::SMEM, stream, a);
    HIP_CHECK_KERNEL();
  };
  using Yes = std::true_type;
  using No = std::false_type;
  if constexpr (FORM == lg::Y) {
    lg::launch_out(a, (unsigned)blocks, stream);
  } else if constexpr (FORM == lg::GLU) {
    lg::launch_glu(a, (unsigned)blocks, stream);
  } else if constexpr (FORM == lg::DW) {
    if (a.parts > 1) launch(Yes{}, Yes{});
    else launch(Yes{}, No{});
  } else {
    if (r2) lg::launch_extra(a, (unsigned)blocks, stream);
    else if (a.parts > 1) launch(No{}, Yes{});
    else if (sum == 2 * gt::STEP) launch(Yes{}, No{});
    else launch(No{}, No{});
  }
  if (a.parts > 1) {
    hipLaunchKernelGGL(add_parts_kernel, dim3((unsigned)(tiles * 4 * (a.height / 32))), dim3(256), 0, stream, a);
    HIP_CHECK_KERNEL();
  }
  return out;
}

}  // namespace

at::Tensor linear_dw(const at::Tensor& g, const at::Tensor& x) {
  TORCH_CHECK(g.dim() == 2 && x.dim() == 2 && g.size(0) == x.size(0), "linear_dw: g [T, N], x [T, K]");
  TORCH_CHECK(g.size(0) > 0 && g.size(1) % 8 == 0 && x.size(1) % 8 == 0, "linear_dw: rows, N%8 == 0, K%8 == 0");
  return run<lg::DW>(g, x, g.size(1), x.size(1), g.size(0));
}

at::Tensor linear_dx(const at::Tensor& g, const at::Tensor& w) {
  TORCH_CHECK(g.dim() == 2 && w.dim() == 2 && g.size(1) == w.size(0), "linear_dx: g [T, N], w [N, K]");
  TORCH_CHECK(w.size(0) > 0 && w.size(0) % (2 * gt::STEP) == 0 && w.size(1) % 8 == 0,
              "linear_dx: N%64 == 0, K%8 == 0");
  return run<lg::DX>(g, w, g.size(0), w.size(1), w.size(0));
}

// the same and t A for t [T, r], A^T [K, r]
at::Tensor linear_dx_extra(const at::Tensor& g, const at::Tensor& w, const at::Tensor& t, const at::Tensor& a_t) {
  TORCH_CHECK(g.dim() == 2 && w.dim() == 2 && g.size(1) == w.size(0), "linear_dx: g [T, N], w [N, K]");
  TORCH_CHECK(w.size(0) > 0 && w.size(0) % (2 * gt::STEP) == 0 && w.size(1) % 8 == 0,
              "linear_dx: N%64 == 0, K%8 == 0");
  for (const at::Tensor* e : {&t, &a_t})
    TORCH_CHECK(e->device() == g.device() && e->scalar_type() == at::kBFloat16 && e->dim() == 2 && e->is_contiguous() &&
                    e->size(1) == t.size(1) && (uintptr_t)e->data_ptr() % 16 == 0, "linear_dx: t [T, r], A^T [K, r]");
  TORCH_CHECK(t.size(1) >= 32 && t.size(1) % 32 == 0 && t.size(0) == g.size(0) && a_t.size(0) == w.size(1),
              "linear_dx: t [T, r], A^T [K, r], r % 32 == 0");
  return run<lg::DX>(g, w, g.size(0), w.size(1), w.size(0), &t, &a_t);
}

// x w^T, or max(x w^T, 0)^2 of the unrounded sums
at::Tensor linear_y(const at::Tensor& x, const at::Tensor& w, bool relu2) {
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1), "linear_y: x [T, K], w [N, K]");
  TORCH_CHECK(w.size(1) >= 4 * gt::STEP && w.size(1) % (2 * gt::STEP) == 0 && w.size(0) % 8 == 0,
              "linear_y: K%64 == 0 and 128 or more, N%8 == 0");
  return run<lg::Y>(x, w, x.size(0), w.size(0), w.size(1), nullptr, nullptr, relu2);
}

// silu(x w^T) (x up^T) of the unrounded sums
at::Tensor linear_glu(const at::Tensor& x, const at::Tensor& w, const at::Tensor& up) {
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1) && up.sizes() == w.sizes(),
              "linear_glu: x [T, K], w and up [I, K]");
  TORCH_CHECK(w.size(1) >= 4 * gt::STEP && w.size(1) % (2 * gt::STEP) == 0 && w.size(0) % 8 == 0 && w.size(0) < (1l << 22),
              "linear_glu: K%64 == 0 and 128 or more, I%8 == 0");
  TORCH_CHECK(up.device() == x.device() && up.is_contiguous() && up.scalar_type() == at::kBFloat16 &&
                  (uintptr_t)up.data_ptr() % 16 == 0, "linear_glu: up as w");
  return run<lg::GLU>(x, w, x.size(0), 2 * w.size(0), w.size(1), nullptr, nullptr, false, &up);
}

// x w^T + scale (x A^T) B^T, A [r, K], B [N, r], r a multiple of 8 up to 64: B's product behind the sums, one rounding. ->
// {it, (x A^T)^T [r rounded up to 32, T to 64] with zeros behind both, which lora_grads reads}. Against the product by
// the faster of kernel and library and lora_forward's pass over it, us: 8192 rows, 4096 -> 28672 1522 -> 1316, 4096 -> 6144
// 338 -> 294, 14336 -> 4096 717 -> 679. Few tiles lose by it, as their sums are cut in parts or not at all, and so
// do few rows of wide layers (ops/linear.py: adapted_own has the rule and what it was fitted to).
std::tuple<at::Tensor, at::Tensor> lora_linear(const at::Tensor& x, const at::Tensor& w, const at::Tensor& A,
                                               const at::Tensor& B, double scale) {
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && A.dim() == 2 && B.dim() == 2 && x.size(1) == w.size(1),
              "lora_linear: x [T, K], w [N, K]");
  const int64_t T = x.size(0), N = w.size(0), K = w.size(1), r = A.size(0);
  TORCH_CHECK(T > 0 && K >= 4 * gt::STEP && K % (2 * gt::STEP) == 0 && N % 64 == 0 && r >= 8 && r <= 64 && r % 8 == 0 &&
                  A.size(1) == K && B.size(0) == N && B.size(1) == r,
              "lora_linear: rows, K%64 == 0 and 128 or more, N%64 == 0, A [r, K], B [N, r], r a multiple of 8 up to 64");
  for (const at::Tensor* t : {&x, &w, &A, &B})
    TORCH_CHECK(t->is_cuda() && t->device() == x.device() && t->scalar_type() == at::kBFloat16 && t->is_contiguous() &&
                    (uintptr_t)t->data_ptr() % 16 == 0, "lora_linear: bf16, whole, at multiples of 16 bytes");
  const c10::DeviceGuard guard(x.device());
  const int64_t R = r <= 32 ? 32 : 64;
  auto t = at::empty({T, R}, x.options()), turned = at::empty({R, (T + 63) / 64 * 64}, x.options());
  lora_down(x, A, r, &t, &turned, scale, 1.);
  return {run<lg::Y>(x, w, T, N, K, &t, &B), turned};
}

// {rows of a tile, parts of the sum} for linear_y of T rows, [N, K]
std::vector<int64_t> linear_y_cut(int64_t T, int64_t N, int64_t K) {
  Args a{};
  a.rows = T;
  a.cols = N;
  a.sum = K;
  cut(lg::Y, a);
  return {a.height, a.parts};
}

// the same for linear_dw (of T rows, [N, K]) or linear_dx
std::vector<int64_t> linear_grad_cut(bool dw, int64_t T, int64_t N, int64_t K) {
  Args a{};
  a.rows = dw ? N : T;
  a.cols = K;
  a.sum = dw ? T : N;
  cut(dw ? lg::DW : lg::DX, a);
  return {a.height, a.parts};
}

}  // namespace amd_ops
