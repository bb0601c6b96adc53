// Grouped GEMM for stacked expert weights (CDNA4, bf16, f32 accumulation): rows of x are sorted by expert,
// expert e owns rows offs[e] .. offs[e+1].
//
//   nt (forward)  y[m, n]  = sum_k x[m, k] w[e(m), n, k]
//   nn (dx)      dx[m, k]  = sum_n g[m, n] w[e(m), n, k], optionally over two pairs of g and w (gate and up):
//                one sum in the accumulators instead of an addition after
//   tn (dw)   dw[e, n, k]  = sum_{m of e} g[m, n] x[m, k]
//
// grouped_tile_kernel has the three for groups of many rows (`tile_cap`): workgroups that stay, tiles of 4 to 8
// times 32 rows by 256 columns, the next tile's operands on their way before a tile ends (gemm_tile.h), dealt
// out by how long they take (grouped_tiles.h).
//
// grouped_gemm_kernel has them for few rows, where a step's time is that of the weights' reads and more
// workgroups of less LDS read more at a time, and for short sums and few columns, where a tile's beginning and end
// are most of it: 8 waves compute BM x 256 of the output, 64 x 64 or 64 x 128 each,
// over steps of 64 of the summed index. What differs is which index of an operand is contiguous: tiles whose
// rows are output rows or columns are read by rows, tiles whose rows are the summed index by columns, with the
// transposing LDS reads (flash_tile.h). So dw takes g and x as they are, and dx takes w as it is. Direct loads
// fill three LDS buffers two steps ahead (256 x 256: two, one ahead, which is what fits), one barrier a step.
// Blocks are dealt to the 8 XCDs in contiguous stretches of the tile list, column tiles of one row tile next to
// each other: an expert's weights and a row tile stay in one L2.
//
// Measured, nt / nn / tn, groups as a random choice fills them, by a workgroup for each tile (nt:
// grouped_gemm_kernel; nn and tn: four waves of 128 x 128 from 512 rows on) -> by grouped_tile_kernel: 65536
// rows, 128 experts, 768 x 2048: 253 / 265 / 270 -> 230 / 227 / 230 us; 2048 x 768: 276 / 232 / 271 -> 252 /
// 210 / 242 us; 19200 rows, 64 experts, 1408 x 2048: 166 / 175 / 197 -> 149 / 129 / 169 us; 16384 rows, 32
// experts, 512 x 1024 (128-row tiles): 32 / 36 / 24 -> 30 / 32 / 24. Since its loads are spread
// evenly (gemm_tile.h) nt of the first takes 220, of the second 235. The products alone are 137 us of the first
// at the 1.5 PFLOP/s that the card holds (its clock falls to 1.2 to 1.9 GHz), its operands and results 150 us
// at 5 TB/s.

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include "common.h"
#include "flash_tile.h"
#include "grouped_tiles.h"
#include "ops_api.h"

namespace amd_ops {

using namespace fa;

namespace {

constexpr int STEP = 64;               // of the summed index

}  // namespace

template <Mode MODE, int BM, int BN, int WAVES, int BUFS>
__global__ __launch_bounds__(64 * WAVES, 1) void grouped_gemm_kernel(const GroupedArgs a) {
  constexpr int WR = BM / 64, WC = WAVES / WR, WN = BN / WC;    // waves down, across; columns of one
  constexpr bool RC = MODE == TN, CC = MODE != NT;              // operand read by columns
  // tiles: [BM][STEP] or, read by columns, [STEP][BM]
  constexpr int RT = RC ? STEP * row_bytes(BM) : BM * row_bytes(STEP);
  constexpr int CT = CC ? STEP * row_bytes(BN) : BN * row_bytes(STEP);
  constexpr int BUF = RT + CT, LOADS = BUF / 1024 / WAVES;
  static_assert(BM % 64 == 0 && WAVES % WR == 0 && (WN == 64 || WN == 128), "wave tiles");
  extern __shared__ __attribute__((aligned(1024))) char smem[];

  // ---- tile of the block
  const int rows_out = MODE == TN ? a.N : 0, cols_out = MODE == NT ? a.N : a.K;
  const int nr = (rows_out + BM - 1) / BM, nc = (cols_out + BN - 1) / BN;
  const int total = MODE == TN ? a.E * nr * nc : (a.n_tiles ? a.n_tiles[0] : a.n_mtiles) * nc;
  const int per = (total + 7) / 8, slot = blockIdx.x >> 3, id = (blockIdx.x & 7) * per + slot;
  if (slot >= per || id >= total) return;
  int e, r0, c0, sum, r_left;          // expert; first row, column; length of the sum; rows left
  const bf16 *rp, *cp, *rp2 = nullptr, *cp2 = nullptr;          // first element of either operand
  if constexpr (MODE == TN) {
    e = id / (nr * nc);
    r0 = id / nc % nr * BM;
    c0 = id % nc * BN;
    const int m0 = a.offs[e];
    sum = a.offs[e + 1] - m0;
    r_left = a.N - r0;
    rp = a.r + (long)m0 * a.N + r0;
    cp = a.c + (long)m0 * a.K + c0;
  } else {
    const int t = id / nc;
    e = a.tile_map[2 * t];
    r0 = a.tile_map[2 * t + 1];
    c0 = id % nc * BN;
    sum = MODE == NT ? a.K : a.N;
    r_left = a.offs[e + 1] - r0;
    rp = a.r + (long)r0 * sum;
    cp = a.c + (long)e * a.N * a.K + (MODE == NT ? (long)c0 * a.K : c0);
    if (MODE == NN && a.r2) {
      rp2 = a.r2 + (long)r0 * sum;
      cp2 = a.c2 + (long)e * a.N * a.K + c0;
    }
  }
  const int c_left = cols_out - c0;
  const unsigned r_rs = (MODE == TN ? a.N : sum) * 2, c_rs = a.K * 2;

  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Waves w and w + 4 share a SIMD: they get different rows and different columns, and a
  // wave without rows or columns of its own (a tile at a group's or the output's end) forms
  // no products, so that half a tile takes half the time. 128 experts x 512 rows, 768 x 2048,
  // nt: 266 -> 259 us (255 in another run); 64 x 281, 1408 x 2048: 175 -> 163. (A choice of 32 or 64 rows in the
  // loop spilled.)
  const int wr = wid / WC, wc = (wid % WC) ^ (wid >= 4 ? WC / 2 : 0);
  const bool live = wr * 64 < r_left && wc * WN < c_left;

  const int once = (sum + STEP - 1) / STEP, steps = MODE == NN && rp2 ? 2 * once : once;
  const unsigned lds = lds_address(smem);
  auto load = [&](int s, unsigned buf) {
    buf += lds;
    const bf16 *r = rp, *c = cp;
    if (MODE == NN && s >= once) {
      r = rp2;
      c = cp2;
      s -= once;
    }
    const int left = sum - s * STEP;   // of the summed index (a multiple of STEP but for tn)
    if constexpr (RC) load_tile<BM, STEP, WAVES>(r + (long)s * STEP * a.N, r_rs, left, buf, r_left / 8);
    else load_tile<STEP, BM, WAVES>(r + s * STEP, r_rs, r_left, buf);
    if constexpr (CC) load_tile<BN, STEP, WAVES>(c + (long)s * STEP * a.K, c_rs, left, buf + RT, c_left / 8);
    else load_tile<STEP, BN, WAVES>(c + s * STEP, c_rs, c_left, buf + RT);
  };
  const unsigned rrow = rows_base<STEP>(), crow = rows_base<STEP>();
  const unsigned rcol = cols_base_natural<BM>(), ccol = cols_base_natural<BN>();

  f32x16_t acc[2][WN / 32];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < WN / 32; ++j) acc[i][j] = zero16();

  unsigned cur = 0, next = BUF, after = 2 * BUF;
  if (steps > 0) load(0, cur);
  if (BUFS == 3 && steps > 1) load(1, next);
  for (int s = 0; s < steps; ++s) {
    if (BUFS == 3 && s + 1 < steps) wait_loads<LOADS>();
    else wait_loads();
    barrier();                         // the step's tiles are there; those of s - 1 are done with
    if (s + BUFS - 1 < steps) load(s + BUFS - 1, BUFS == 3 ? after : next);
    if constexpr (MODE == TN) {
      // rows of the next expert, or beyond the end: clamped by the load, zeroed here
      const int left = sum - s * STEP;
      if (left < STEP) {
        for (int i = threadIdx.x; i < (STEP - left) * (row_bytes(BM) / 16); i += 64 * WAVES)
          *reinterpret_cast<uint4*>(smem + cur + left * row_bytes(BM) + i * 16) = uint4{0, 0, 0, 0};
        barrier();
      }
    }
    if (live)
#pragma unroll
      for (int ch = 0; ch < STEP / 16; ++ch) {
        bf16x8_t rf[2], cf[WN / 32];
#pragma unroll
        for (int i = 0; i < 2; ++i)
          rf[i] = RC ? read_cols_natural<BM>(smem, cur, rcol, ch, wr * 2 + i)
                     : read_rows<STEP>(smem, cur + wr * 64 * row_bytes(STEP), rrow, i, ch);
#pragma unroll
        for (int j = 0; j < WN / 32; ++j)
          cf[j] = CC ? read_cols_natural<BN>(smem, cur + RT, ccol, ch, wc * (WN / 32) + j)
                     : read_rows<STEP>(smem, cur + RT + wc * WN * row_bytes(STEP), crow, j, ch);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < WN / 32; ++j) acc[i][j] = mma(cf[j], rf[i], acc[i][j]);
      }
    const unsigned t = cur;
    cur = next;
    next = BUFS == 3 ? after : t;
    after = t;
  }
  barrier();                           // the buffers are the waves' output tiles now

  char* mine = smem + wid * 32 * row_bytes(WN);
  const int cw = c0 + wc * WN, cols = min(cols_out - cw, WN);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int rw = wr * 64 + i * 32;   // row of the block's tile
    const long row = MODE == TN ? (long)e * a.N + r0 + rw : r0 + rw;
    if (cols > 0)
      store_rows<WN>(acc[i], 1.f, mine, a.out + row * cols_out + cw, cols_out, r_left - rw, cols / 8);
  }
}

// The same by the tiles of gemm_tile.h.
template <Mode MODE>
__global__ __launch_bounds__(gt::THREADS, 1) void grouped_tile_kernel(const GroupedArgs a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  GroupedTiles<MODE> tiles(a, smem);
  constexpr bool ROWS = MODE == NT || MODE == GLU;
  const gt::Shape shape{2u * (ROWS ? a.K : a.N), 2u * a.K, 2u * (ROWS ? a.N : a.K)};
  gt::Run<MODE == TN, !ROWS, GroupedTiles<MODE>, MODE == TN, false, false, false, MODE == GLU, MODE == GLU>(tiles, shape, smem)();
}

// Offsets and (expert, first row) tiles of the groups, from counts on the device, so that
// routing never waits for the host. One workgroup: thread t sums a stretch of experts, a
// scan over the threads gives every stretch its first row and tile. (A single thread took
// 26 us for 128 experts, now 11 with the launch.)
__global__ __launch_bounds__(256) void build_group_plan_kernel(const int* __restrict__ counts, int E,
                                                               int* __restrict__ offs,
                                                               int* __restrict__ tile_map,
                                                               int* __restrict__ n_tiles, int bm,
                                                               int capacity) {
  __shared__ int rows[256], tiles[256];
  const int t = threadIdx.x, per = (E + 255) / 256, e0 = min(t * per, E), e1 = min(e0 + per, E);
  int r = 0, n = 0;
  for (int e = e0; e < e1; ++e) {
    r += counts[e];
    n += (counts[e] + bm - 1) / bm;
  }
  rows[t] = r;
  tiles[t] = n;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const int rr = t >= off ? rows[t - off] : 0, nn = t >= off ? tiles[t - off] : 0;
    __syncthreads();
    rows[t] += rr;
    tiles[t] += nn;
    __syncthreads();
  }
  if (t == 255) n_tiles[0] = min(tiles[255], capacity);
  if (t == 0) offs[0] = 0;
  r = rows[t] - r;
  n = tiles[t] - n;
  for (int e = e0; e < e1; ++e) {
    for (int m = 0; m < counts[e]; m += bm, ++n)
      if (n < capacity) {
        tile_map[2 * n] = e;
        tile_map[2 * n + 1] = r + m;
      }
    r += counts[e];
    offs[e + 1] = r;
  }
}

std::tuple<at::Tensor, at::Tensor, at::Tensor> build_group_plan(
    const at::Tensor& counts, int64_t M, int64_t bm) {
  TORCH_CHECK(counts.is_cuda() && counts.scalar_type() == at::kInt,
              "build_group_plan: counts int32 on GPU");
  const int E = counts.size(0);
  const long max_tiles = M / bm + E + 1;
  auto opts = counts.options();
  auto offs = at::empty({E + 1}, opts);
  auto tile_map = at::empty({max_tiles, 2}, opts);
  auto n_tiles = at::empty({1}, opts);
  auto stream = c10::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(build_group_plan_kernel, dim3(1), dim3(256), 0, stream.stream(),
                     counts.data_ptr<int>(), E, offs.data_ptr<int>(),
                     tile_map.data_ptr<int>(), n_tiles.data_ptr<int>(), (int)bm, (int)max_tiles);
  HIP_CHECK_KERNEL();
  return {offs, tile_map, n_tiles};
}

namespace {

// Rows of grouped_tile_kernel's tiles at most, or 0 where grouped_gemm_kernel is the faster one; M rows in E
// groups, weights [E, N, K]. 9210 shapes each of nt, nn and tn (2 to 512 groups of 16 to 2000 rows on average,
// filled at random or unequally, widths and sums of 128 to 4096) take 0.87, 0.81 and 0.84 of the time where the
// rule has the tiles; 1% of these more than 1.05, 1.24 at most. What decides is how many rows an
// expert's weights serve, whether the tiles fill the chip's rounds, and what a tile costs beside its products:
//   tn      from 320 rows a group on (0.75 to 1.01); from 128 on with two rounds of tiles (0.81 to 1.02; with
//           fewer 1.0 to 1.2). Not with 128 columns, half of a tile's (1.07 in the mean, to 1.48)
//   nt, nn  from 512 rows on, tiles of 128 for up to half a round (0.65 to 1.0); from 200 rows on (nn with sums from 768
//           on: 128) with 168 to 256 tiles of 256 rows (0.55 to 0.9); from 256 (nt) with 360 and more (0.8 to 1.0).
//           Between them is a short second round (1.0 to 1.15), below them are idle CUs (1.1 to 1.5)
//   nn      also otherwise from 80 rows on, tiles of 128 (0.8 to 1.05): sums from 1024 on (768: 1.0 to 1.2), and with
//           128 columns from 2048 on
//   nt, nn  no sums below 512 and no 128 columns with more tiles than half a round (sums of 128 1.14 in the mean, to 2.06;
//           of 256 1.05, to 1.8; 128 columns 1.07 to 1.13, to 2.0): a tile's beginning and stores are most of it,
//           and the other kernel's workgroups overlap them. With fewer tiles sums from 256 on (0.83 to 0.96)
//   any     of small weights, up to 2^20, no more than 256 groups, and more than 128 from 320 rows on: every workgroup
//           sorts all groups (256 of 130 to 200 rows: nt 1.14, nn 1.02, tn 0.96; 512: 1.16, 1.18, 1.02; but with
//           weights of 1408 x 2048 and more 0.9, 0.8 and 0.85)
template <Mode MODE>
int tile_cap(long M, long E, long N, long K) {
  const long cols = MODE == NT ? N : K, sum = MODE == NT ? K : N, rows = M / std::max(E, 1l);
  // the table of groups, 32-bit addresses within a tile
  if (E < 1 || E > MAX_GROUPS || std::max(N, K) >= (1 << 23)) return 0;
  if (E > 128 && N * K <= (1l << 20) && (E > 256 || rows < 320)) return 0;
  const long nc = (cols + gt::TILE - 1) / gt::TILE;
  if (MODE == TN) {
    if (K < 256 && N >= 256) return 0;
    return rows >= 320 || (rows >= 128 && E * ((N + gt::TILE - 1) / gt::TILE) * nc >= 512) ? 256 : 0;
  }
  // parts of groups that are not all of one size
  const auto parts = [&](long pct) { return (M * pct / 100 + E * 256 - 1) / (E * 256); };
  const long tiles = E * nc * (parts(95) + parts(101) + parts(107)) / 3;
  const bool few = tiles <= 128, long_sum = sum >= 512, wide = cols >= 256;
  if (sum < 256 || (few ? !long_sum && !wide : !long_sum || !wide)) return 0;
  if (rows >= 512) return few ? 128 : 256;
  const bool fills = (tiles >= 168 && tiles <= 256) || tiles >= 360;
  if (MODE == NT) return rows >= (tiles >= 360 ? 256 : 200) && fills ? 256 : 0;
  if (rows >= (sum >= 768 ? 128 : 200) && fills) return 256;
  return rows >= (tiles < 168 ? 80 : 128) && sum >= (wide ? 1024 : 2048) ? 128 : 0;
}

// by grouped_tile_kernel, or by grouped_gemm_kernel with tiles of `tile` rows
template <Mode MODE>
void launch(GroupedArgs& a, int64_t tile) {
  const auto stream = c10::hip::getCurrentHIPStream().stream();
  // its loads take whole pieces of 16 bytes
  const uintptr_t at = (uintptr_t)a.r | (uintptr_t)a.c | (uintptr_t)a.r2 | (uintptr_t)a.c2;
  a.cap = at % 16 ? 0 : tile_cap<MODE>(a.M, a.E, a.N, a.K);
  if (a.cap) {
    hipLaunchKernelGGL((grouped_tile_kernel<MODE>), dim3((unsigned)gt::workgroups()), dim3(gt::THREADS),
                       GroupedTiles<MODE>::SMEM, stream, a);
    HIP_CHECK_KERNEL();
    return;
  }
  const int nc = ((MODE == NT ? a.N : a.K) + 255) / 256;
  const long tiles = MODE == TN ? (long)a.E * ((a.N + 255) / 256) * nc : (long)a.n_mtiles * nc;
  TORCH_CHECK(tiles < (1l << 31) - 8, "grouped_gemm: too many tiles");
  // the stretches of the 8 XCDs are rounded up: up to 7 workgroups beyond the tiles
  const dim3 grid((unsigned)((tiles + 7) / 8 * 8));
  auto eight = [&](auto bm_, auto bufs_) {
    constexpr int BM = decltype(bm_)::value, BUFS = decltype(bufs_)::value;
    constexpr int rt = MODE == TN ? STEP * row_bytes(BM) : BM * row_bytes(STEP);
    constexpr int ct = MODE != NT ? STEP * row_bytes(256) : 256 * row_bytes(STEP);
    constexpr int smem = std::max(BUFS * (rt + ct), 8 * 32 * row_bytes(BM / 2));
    hipLaunchKernelGGL((grouped_gemm_kernel<MODE, BM, 256, 8, BUFS>), grid, dim3(512), smem, stream, a);
  };
  if constexpr (MODE != TN)
    if (tile == 128) {
      eight(std::integral_constant<int, 128>{}, std::integral_constant<int, 3>{});
      HIP_CHECK_KERNEL();
      return;
    }
  eight(std::integral_constant<int, 256>{}, std::integral_constant<int, 2>{});
  HIP_CHECK_KERNEL();
}

GroupedArgs grouped_args(const at::Tensor& r, const at::Tensor& c, at::Tensor& out,
                         const at::Tensor& offs) {
  TORCH_CHECK(r.is_cuda() && r.is_contiguous() && c.is_contiguous() && r.scalar_type() == at::kBFloat16 &&
                  c.scalar_type() == at::kBFloat16, "grouped_gemm: contiguous bf16 operands");
  TORCH_CHECK(offs.scalar_type() == at::kInt && offs.is_contiguous(), "grouped_gemm: offs int32");
  GroupedArgs a{};
  a.r = reinterpret_cast<const bf16*>(r.data_ptr());
  a.c = reinterpret_cast<const bf16*>(c.data_ptr());
  a.out = reinterpret_cast<bf16*>(out.data_ptr());
  a.offs = offs.data_ptr<int>();
  a.M = r.size(0);
  return a;
}

void set_tiles(GroupedArgs& a, const at::Tensor& w, const at::Tensor& offs, const at::Tensor& tile_map,
               const std::optional<at::Tensor>& n_tiles) {
  TORCH_CHECK(tile_map.scalar_type() == at::kInt && tile_map.is_contiguous(), "tile_map int32 [n, 2]");
  TORCH_CHECK(offs.numel() == w.size(0) + 1, "offs [E + 1]");
  a.tile_map = tile_map.data_ptr<int>();
  a.n_tiles = n_tiles.has_value() ? n_tiles->data_ptr<int>() : nullptr;
  a.n_mtiles = tile_map.size(0);
  a.E = w.size(0);
  a.N = w.size(1);
  a.K = w.size(2);
}

}  // namespace

at::Tensor grouped_gemm_nt(const at::Tensor& x, const at::Tensor& w,
                           const at::Tensor& offs, const at::Tensor& tile_map,
                           const std::optional<at::Tensor>& n_tiles, int64_t bm) {
  TORCH_CHECK(x.dim() == 2 && w.dim() == 3 && x.size(1) == w.size(2), "grouped_gemm_nt: x [M,K], w [E,N,K]");
  TORCH_CHECK(w.size(2) % STEP == 0 && w.size(1) % 128 == 0, "need K%64==0, N%128==0");
  TORCH_CHECK(bm == 128 || bm == 256, "grouped_gemm_nt: tiles of 128 or 256 rows");
  auto y = at::empty({x.size(0), w.size(1)}, x.options());
  if (tile_map.size(0) == 0 || x.size(0) == 0) return y;
  auto a = grouped_args(x, w, y, offs);
  set_tiles(a, w, offs, tile_map, n_tiles);
  launch<NT>(a, bm);
  return y;
}

// {x w^T, x up^T, silu(the one) the other} of the groups. By the tiles of gemm_tile.h x is read once for both and the
// activation is no pass of its own. The tiles are nt's of twice the columns, and so is the
// rule. us, two products and swiglu -> here: 65536 rows, 128 experts, 768 x 2048 494 -> 430; 18018 rows, 64, 1408 x 2048
// 323 -> 276; 291 shapes (4 to 128 groups of 60 to 2000 rows, 384 to 2048 columns, sums of 512 to 4096) 0.82 of the time
// in the mean, 4 of them above 1.02, 1.16 at most.
std::tuple<at::Tensor, at::Tensor, at::Tensor> grouped_glu(const at::Tensor& x, const at::Tensor& w, const at::Tensor& up,
                                                           const at::Tensor& offs, const at::Tensor& tile_map,
                                                           const std::optional<at::Tensor>& n_tiles, int64_t bm) {
  TORCH_CHECK(x.dim() == 2 && w.dim() == 3 && x.size(1) == w.size(2) && up.sizes() == w.sizes(),
              "grouped_glu: x [M,K], w and up [E,N,K]");
  TORCH_CHECK(up.is_cuda() && up.device() == w.device() && up.is_contiguous() && up.scalar_type() == at::kBFloat16,
              "grouped_glu: contiguous bf16 operands");
  const long M = x.size(0), E = w.size(0), N = w.size(1), K = w.size(2);
  const uintptr_t at = (uintptr_t)x.data_ptr() | (uintptr_t)w.data_ptr() | (uintptr_t)up.data_ptr();
  const int cap = at % 16 || N % 128 || K % STEP || N >= (1 << 22) ? 0 : tile_cap<NT>(M, E, 2 * N, K);
  if (!cap || tile_map.size(0) == 0 || M == 0) {
    auto g = grouped_gemm_nt(x, w, offs, tile_map, n_tiles, bm), u = grouped_gemm_nt(x, up, offs, tile_map, n_tiles, bm);
    return {g, u, g.numel() ? swiglu_fwd(g, u) : at::empty_like(g)};
  }
  auto g = at::empty({M, N}, x.options()), u = at::empty_like(g), h = at::empty_like(g);
  auto a = grouped_args(x, w, h, offs);
  set_tiles(a, w, offs, tile_map, n_tiles);
  a.up = reinterpret_cast<const bf16*>(up.data_ptr());
  a.one = reinterpret_cast<bf16*>(g.data_ptr());
  a.other = reinterpret_cast<bf16*>(u.data_ptr());
  a.cap = cap;
  hipLaunchKernelGGL((grouped_tile_kernel<GLU>), dim3((unsigned)gt::workgroups()), dim3(gt::THREADS), GroupedTiles<GLU>::SMEM,
                     c10::hip::getCurrentHIPStream().stream(), a);
  HIP_CHECK_KERNEL();
  return {g, u, h};
}

static at::Tensor nn(const at::Tensor& g, const at::Tensor& w, const at::Tensor* g2, const at::Tensor* w2,
                     const at::Tensor& offs, const at::Tensor& tile_map,
                     const std::optional<at::Tensor>& n_tiles, int64_t bm) {
  TORCH_CHECK(g.dim() == 2 && w.dim() == 3 && g.size(1) == w.size(1), "grouped_gemm_nn: g [M,N], w [E,N,K]");
  TORCH_CHECK(bm == 128 || bm == 256, "grouped_gemm_nn: tiles of 128 or 256 rows");
  TORCH_CHECK(w.size(1) % STEP == 0 && w.size(2) % 128 == 0, "need N%64==0, K%128==0");
  auto dx = at::empty({g.size(0), w.size(2)}, g.options());
  if (tile_map.size(0) == 0 || g.size(0) == 0) return dx;
  auto a = grouped_args(g, w, dx, offs);
  if (g2) {
    TORCH_CHECK(g2->sizes() == g.sizes() && w2->sizes() == w.sizes(), "grouped_gemm_nn2: two equal pairs");
    auto b = grouped_args(*g2, *w2, dx, offs);
    a.r2 = b.r;
    a.c2 = b.c;
  }
  set_tiles(a, w, offs, tile_map, n_tiles);
  launch<NN>(a, bm);
  return dx;
}

at::Tensor grouped_gemm_nn(const at::Tensor& g, const at::Tensor& w,
                           const at::Tensor& offs, const at::Tensor& tile_map,
                           const std::optional<at::Tensor>& n_tiles, int64_t bm) {
  return nn(g, w, nullptr, nullptr, offs, tile_map, n_tiles, bm);
}

at::Tensor grouped_gemm_nn2(const at::Tensor& g1, const at::Tensor& w1, const at::Tensor& g2,
                            const at::Tensor& w2, const at::Tensor& offs, const at::Tensor& tile_map,
                            const std::optional<at::Tensor>& n_tiles, int64_t bm) {
  return nn(g1, w1, &g2, &w2, offs, tile_map, n_tiles, bm);
}

// tile_cap of grouped_gemm_nt, _nn and _tn (mode 0, 1, 2)
int64_t grouped_gemm_cap(int64_t mode, int64_t M, int64_t E, int64_t N, int64_t K) {
  return mode == 0 ? tile_cap<NT>(M, E, N, K) : mode == 1 ? tile_cap<NN>(M, E, N, K) : tile_cap<TN>(M, E, N, K);
}

at::Tensor grouped_gemm_tn(const at::Tensor& g, const at::Tensor& x, const at::Tensor& offs, int64_t E) {
  TORCH_CHECK(g.dim() == 2 && x.dim() == 2 && g.size(0) == x.size(0) && offs.numel() == E + 1,
              "grouped_gemm_tn: g [M,N], x [M,K], offs [E+1]");
  TORCH_CHECK(g.size(1) % 128 == 0 && x.size(1) % 128 == 0, "need N%128==0, K%128==0");
  auto dw = at::empty({E, g.size(1), x.size(1)}, g.options());
  if (dw.numel() == 0) return dw;
  auto a = grouped_args(g, x, dw, offs);
  a.E = E;
  a.N = g.size(1);
  a.K = x.size(1);
  launch<TN>(a, 256);
  return dw;
}

}  // namespace amd_ops
