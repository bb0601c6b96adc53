// x w^T and its gradients for small layers, bf16 with f32 accumulation (gfx950):
//
//   nt   y[t, n] = sum_k x[t, k] w[n, k]
//   nn  dx[t, k] = sum_n g[t, n] w[n, k]
//   tn  dw[n, k] = sum_t g[t, n] x[t, k]
//
// These are a few us each, most of them beginning and end, and what they wait for is the host, which takes 28 us to
// call one of the library's and 4 for one of these. A workgroup is 2 x 2 waves on a tile of 64 x 64 or, where there
// are many tiles, 128 x 128; steps of 64 of the summed index come straight to LDS, the operands as they are (read by
// rows, or by columns with the transposing reads: flash_tile.h). Two steps are under way (128: one, two workgroups to a
// CU). Where few tiles have long sums these are cut into parts, kept in 32 bits and added up in their order. x w^T of few
// rows is another kernel's.
//
// us, library -> here, captured, so that neither waits for the host: nt 256 x 256 x 256 11.7 -> 3.5, 256 x 1024 x 256
// 4.3 -> 3.5, 1000 x 1536 x 2048 13.1 -> 14; nn 256 x 512 x 256 18.8 -> 4.4, 500 x 1536 x 2048 11.3 -> 9, 1000 x 3584 x
// 1024 20.9 -> 18; tn 256 x 1024 x 256 6.2 -> 3.5, 500 x 1536 x 2048 14 -> 8, 2000 x 1536 x 2048 34 -> 25.
#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <cmath>

#include "common.h"
#include "flash_tile.h"
#include "gemm_tile.h"
#include "ops_api.h"

namespace amd_ops {
namespace {

using namespace fa;

constexpr int STEP = 64, WAVES = 4;    // of the summed index; 2 x 2 waves a workgroup
constexpr unsigned NOWHERE = 0xfffffff0u, REACH = 0xffffff00u;
// Up to so many rows x w^T is gemv.hip's, which reads the weights once: 0.65 of the library's time in the mean, captured,
// above 1.05 for one shape in a hundred; the tiles here 0.96 and two in five, up to 1.67. From 17 to 32 rows 0.92 and 0.93,
// then 1.3 and more against 0.85 (2901 shapes of 1 to 64 rows, 256 to 32768 columns and sums).
constexpr int64_t FEW = 16;

struct Args {
  const bf16 *r, *c;
  bf16* out;
  float* part;                         // [part][tile][wave][accumulators], 32 bits
  int rows, cols, sum;
  int parts, per;                      // parts of the sum, and how much of it each but the last has
};

// One operand's tile, [EDGE][STEP] or, read by columns, [STEP][EDGE]. What lies outside of the output or behind the
// sum is zeros.
template <bool COLS, int EDGE>
struct Side {
  static constexpr int D = COLS ? EDGE : STEP, ROWS = COLS ? STEP : EDGE, RB = row_bytes(D);
  static constexpr int BYTES = ROWS * RB, LOADS = BYTES / 1024 / WAVES, PER = 1024 / RB;
  unsigned off[LOADS];
  const char* base;
  unsigned ld;

  __device__ __forceinline__ int row(int i, int lane, int wid) const { return (i * WAVES + wid) * PER + lane / (RB / 16); }
  __device__ __forceinline__ int chunk(int row, int lane) const { return (lane % (RB / 16)) ^ swz<D>(row); }
  __device__ __forceinline__ void init(const bf16* p, unsigned ld_, int edge, int lane, int wid) {
    base = reinterpret_cast<const char*>(p);
    ld = ld_;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int r = row(i, lane, wid), c = chunk(r, lane);
      off[i] = (COLS ? c * 8 : r) < edge ? r * ld + c * 16 : NOWHERE;
    }
  }
  __device__ __forceinline__ void load(unsigned lds, int left, int lane, int wid) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      unsigned o = off[i];
      if (left < STEP) {               // uniform
        const int r = row(i, lane, wid);
        if ((COLS ? r : chunk(r, lane) * 8) >= left) o = NOWHERE;
      }
      gt::load_lds(lds, (i * WAVES + wid) * 1024, o, base, REACH);
    }
    base += COLS ? (unsigned long)ld * STEP : 2ul * STEP;
  }
};

template <bool RC, bool CC, int BM, int BN, int BUFS, bool PARTS>
__global__ __launch_bounds__(256) void small_kernel(const Args a) {
  constexpr int WM = BM / 2, WN = BN / 2, RT = Side<RC, BM>::BYTES, CT = Side<CC, BN>::BYTES, BUF = RT + CT;
  constexpr int LOADS = Side<RC, BM>::LOADS + Side<CC, BN>::LOADS;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nc = (a.cols + BN - 1) / BN, nr = (a.rows + BM - 1) / BM;
  const int part = PARTS ? blockIdx.x / (nr * nc) : 0, tile = blockIdx.x - part * nr * nc;
  const int r0 = tile / nc * BM, c0 = tile % nc * BN, from = part * a.per;
  const int sum = PARTS ? min(a.per, a.sum - from) : a.sum;
  Side<RC, BM> R;
  Side<CC, BN> C;
  R.init(RC ? a.r + (long)from * a.rows + r0 : a.r + (long)r0 * a.sum + from, 2u * (RC ? a.rows : a.sum), a.rows - r0, lane, wid);
  C.init(CC ? a.c + (long)from * a.cols + c0 : a.c + (long)c0 * a.sum + from, 2u * (CC ? a.cols : a.sum), a.cols - c0, lane, wid);
  const unsigned lds = lds_address(smem);
  const int steps = (sum + STEP - 1) / STEP;
  auto load = [&](int s, unsigned buf) __attribute__((always_inline)) {
    R.load(lds + buf, sum - s * STEP, lane, wid);
    C.load(lds + buf + RT, sum - s * STEP, lane, wid);
  };
  const int wr = wid >> 1, wc = wid & 1;
  const unsigned rrow = rows_base<STEP>(), rcol = cols_base_natural<BM>(), ccol = cols_base_natural<BN>();
  f32x16_t acc[WM / 32][WN / 32];
#pragma unroll
  for (int i = 0; i < WM / 32; ++i)
#pragma unroll
    for (int j = 0; j < WN / 32; ++j) acc[i][j] = zero16();
  unsigned cur = 0, next = BUF, after = 2 * BUF;
  load(0, cur);
  if (BUFS == 3 && steps > 1) load(1, next);
#pragma unroll 1
  for (int s = 0; s < steps; ++s) {
    if (BUFS == 3 && s + 1 < steps) wait_loads<LOADS>();
    else wait_loads();
    barrier();                         // the step's tiles are there; those of s - 1 are done with
    if (s + BUFS - 1 < steps) load(s + BUFS - 1, BUFS == 3 ? after : next);
#pragma unroll
    for (int ch = 0; ch < STEP / 16; ++ch) {
      bf16x8_t rf[WM / 32], cf[WN / 32];
#pragma unroll
      for (int i = 0; i < WM / 32; ++i)
        rf[i] = RC ? read_cols_natural<BM>(smem, cur, rcol, ch, wr * (WM / 32) + i)
                   : read_rows<STEP>(smem, cur + wr * WM * row_bytes(STEP), rrow, i, ch);
#pragma unroll
      for (int j = 0; j < WN / 32; ++j)
        cf[j] = CC ? read_cols_natural<BN>(smem, cur + RT, ccol, ch, wc * (WN / 32) + j)
                   : read_rows<STEP>(smem, cur + RT + wc * WN * row_bytes(STEP), rrow, j, ch);
#pragma unroll
      for (int i = 0; i < WM / 32; ++i)
#pragma unroll
        for (int j = 0; j < WN / 32; ++j) acc[i][j] = mma(cf[j], rf[i], acc[i][j]);
    }
    const unsigned t = cur;
    cur = next;
    next = BUFS == 3 ? after : t;
    after = t;
  }
  if constexpr (PARTS) {
    float* to = a.part + ((long)blockIdx.x * WAVES + wid) * (WM * WN) + lane * 4;
#pragma unroll
    for (int i = 0; i < WM / 32; ++i)
#pragma unroll
      for (int j = 0; j < WN / 32; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<float4*>(to + ((i * (WN / 32) + j) * 4 + q) * 256) =
              float4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
  } else {
    barrier();                         // the buffers are the waves' output tiles now
    char* mine = smem + wid * 32 * row_bytes(WN);
    const int cw = c0 + wc * WN;
#pragma unroll
    for (int i = 0; i < WM / 32; ++i) {
      const int rw = r0 + wr * WM + i * 32;
      if (cw < a.cols)
        store_rows<WN>(acc[i], 1.f, mine, a.out + (long)rw * a.cols + cw, a.cols, a.rows - rw, min(a.cols - cw, WN) / 8);
    }
  }
}

// the parts' sums, in their order
template <int BM, int BN>
__global__ __launch_bounds__(256) void add_small_kernel(const Args a) {
  constexpr int WM = BM / 2, WN = BN / 2;
  __shared__ __attribute__((aligned(16))) char smem[WAVES * 32 * row_bytes(WN)];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nc = (a.cols + BN - 1) / BN, nr = (a.rows + BM - 1) / BM;
  const int i = blockIdx.x % (WM / 32), tile = blockIdx.x / (WM / 32);
  const int r0 = tile / nc * BM + (wid >> 1) * WM + i * 32, c0 = tile % nc * BN + (wid & 1) * WN;
  if (r0 >= a.rows || c0 >= a.cols) return;
  f32x16_t acc[WN / 32];
#pragma unroll
  for (int j = 0; j < WN / 32; ++j) acc[j] = zero16();
  const float* from = a.part + ((long)tile * WAVES + wid) * (WM * WN) + lane * 4;
  for (int p = 0; p < a.parts; ++p, from += (long)nr * nc * WAVES * (WM * WN))
#pragma unroll
    for (int j = 0; j < WN / 32; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float4 v = *reinterpret_cast<const float4*>(from + ((i * (WN / 32) + j) * 4 + q) * 256);
        acc[j][4 * q] += v.x;
        acc[j][4 * q + 1] += v.y;
        acc[j][4 * q + 2] += v.z;
        acc[j][4 * q + 3] += v.w;
      }
  store_rows<WN>(acc, 1.f, smem + wid * 32 * row_bytes(WN), a.out + (long)r0 * a.cols + c0, a.cols, a.rows - r0,
                 min(a.cols - c0, WN) / 8);
}

template <bool RC, bool CC, int BM, int BN>
void launch(const Args& a, hipStream_t stream) {
  constexpr int BUF = Side<RC, BM>::BYTES + Side<CC, BN>::BYTES, BUFS = BM == 128 ? 2 : 3;
  const long tiles = (long)((a.rows + BM - 1) / BM) * ((a.cols + BN - 1) / BN);
  if (a.parts > 1) {
    hipLaunchKernelGGL((small_kernel<RC, CC, BM, BN, BUFS, true>), dim3((unsigned)(tiles * a.parts)), dim3(256), BUFS * BUF,
                       stream, a);
    HIP_CHECK_KERNEL();
    hipLaunchKernelGGL((add_small_kernel<BM, BN>), dim3((unsigned)(tiles * (BM / 64))), dim3(256), 0, stream, a);
  } else {
    hipLaunchKernelGGL((small_kernel<RC, CC, BM, BN, BUFS, false>), dim3((unsigned)tiles), dim3(256), BUFS * BUF, stream, a);
  }
  HIP_CHECK_KERNEL();
}

// us that tiles of 64 or 128 and the sums in `parts` take: a workgroup's start, and a step's time, which grows with
// the workgroups of the fullest CU. Fitted to 162 shapes of 128 to 8000 rows, 256 to 4096 columns, 8 ways each:
// off by 10% (rms), the choice by it by 1% in the mean from the best.
float predicted(long rows, long cols, long sum, int edge, int parts) {
  struct Fit {
    float start, step, shared, each, add, add_mb;
  };
  const Fit f = edge == 64 ? Fit{2.1f, .28f, .21f, .28f, 1.9f, .21f} : Fit{2.5f, .59f, .37f, .8f, 3.7f, .3f};
  const long per = (sum + STEP * parts - 1) / (STEP * parts) * STEP;
  parts = (int)((sum + per - 1) / per);
  const float fill = (float)((rows + edge - 1) / edge * ((cols + edge - 1) / edge) * parts) / 256.f;
  const float most = fill <= 1.f ? 1.f : fill < 4.f ? std::ceil(fill) : fill;
  const float t = f.start + per / STEP * (f.step + f.shared * (most - 1.f)) + f.each * most;
  return parts == 1 ? t : t + f.add + f.add_mb * 4e-6f * rows * cols * parts;
}

template <bool RC, bool CC>
at::Tensor product(const at::Tensor& r, const at::Tensor& c, int64_t rows, int64_t cols, int64_t sum) {
  const c10::DeviceGuard guard(r.device());
  auto out = at::empty({rows, cols}, r.options());
  Args a{reinterpret_cast<const bf16*>(r.data_ptr()), reinterpret_cast<const bf16*>(c.data_ptr()),
         reinterpret_cast<bf16*>(out.data_ptr()), nullptr, (int)rows, (int)cols, (int)sum, 0, 0};
  const auto [edge, parts] = small_cut(rows, cols, sum);
  a.per = (int)((sum + STEP * parts - 1) / (STEP * parts) * STEP);
  a.parts = (int)((sum + a.per - 1) / a.per);
  at::Tensor part;
  if (a.parts > 1) {
    part = at::empty({(rows + edge - 1) / edge * ((cols + edge - 1) / edge) * edge * edge * a.parts}, r.options().dtype(at::kFloat));
    a.part = part.data_ptr<float>();
  }
  const auto stream = c10::hip::getCurrentHIPStream().stream();
  if (edge == 128) launch<RC, CC, 128, 128>(a, stream);
  else launch<RC, CC, 64, 64>(a, stream);
  return out;
}

void check(const at::Tensor& a, const at::Tensor& b, const char* name) {
  TORCH_CHECK(a.is_cuda() && a.device() == b.device() && a.dim() == 2 && b.dim() == 2 && a.is_contiguous() && b.is_contiguous() &&
                  a.scalar_type() == at::kBFloat16 && b.scalar_type() == at::kBFloat16 && (uintptr_t)a.data_ptr() % 16 == 0 &&
                  (uintptr_t)b.data_ptr() % 16 == 0, name, ": two whole bf16 matrices on one GPU, at multiples of 16 bytes");
}

}  // namespace

// {rows and columns of a tile, parts of the sum}
std::tuple<int64_t, int64_t> small_cut(int64_t rows, int64_t cols, int64_t sum) {
  int64_t edge = 64, parts = 1;
  float least = predicted(rows, cols, sum, 64, 1);
  for (const int e : {64, 128})
    for (const int p : {1, 2, 4, 8}) {
      const float t = predicted(rows, cols, sum, e, p);
      if (sum < 128 * p || t >= least) continue;       // a part has two steps or more
      least = t;
      edge = e;
      parts = p;
    }
  return {edge, parts};
}

bool small_takes(int64_t T, int64_t N, int64_t K) {
  // a tile's addresses are 32 bits: 128 rows of 2^23; a grid is too
  return T > 0 && N > 0 && K > 0 && N % 8 == 0 && K % 8 == 0 && std::max({T, N, K}) < (1l << 23) &&
         T * N < (1l << 40) && N * K < (1l << 40) && T * K < (1l << 40);
}

at::Tensor small_nt(const at::Tensor& x, const at::Tensor& w) {
  check(x, w, "small_nt");
  TORCH_CHECK(x.size(1) == w.size(1) && small_takes(x.size(0), w.size(0), w.size(1)), "small_nt: x [T, K], w [N, K], N%8 == 0, K%8 == 0");
  if (x.size(0) <= FEW) {
    const c10::DeviceGuard guard(x.device());
    return gemm_skinny_bf16(x, w, false, false, 0);
  }
  return product<false, false>(x, w, x.size(0), w.size(0), w.size(1));
}
at::Tensor small_nn(const at::Tensor& g, const at::Tensor& w) {
  check(g, w, "small_nn");
  TORCH_CHECK(g.size(1) == w.size(0) && small_takes(g.size(0), w.size(0), w.size(1)), "small_nn: g [T, N], w [N, K], N%8 == 0, K%8 == 0");
  return product<false, true>(g, w, g.size(0), w.size(1), w.size(0));
}
at::Tensor small_tn(const at::Tensor& g, const at::Tensor& x) {
  check(g, x, "small_tn");
  TORCH_CHECK(g.size(0) == x.size(0) && small_takes(g.size(0), g.size(1), x.size(1)), "small_tn: g [T, N], x [T, K], N%8 == 0, K%8 == 0");
  return product<true, true>(g, x, g.size(1), x.size(1), g.size(0));
}

}  // namespace amd_ops
