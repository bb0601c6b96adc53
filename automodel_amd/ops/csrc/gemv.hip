// Linear layers of decode steps: y[B, N] = x[B, K] W[N, K]^T for few rows x.
//
// The weights are read once and are all the traffic there is; both kernels are
// bound by how many of their loads are in flight. Up to 2 rows (4 with a bias) a
// wave takes a row of W and its lanes run along K; above that the matrix cores
// take 16 rows of W against 16 rows of x per instruction, since a dot product
// per row of x would cost more than the load (4 rows, 14336 x 4096: 27 us against
// 21 us), to 16 rows with the kernel of gemm_stream.h where K % 128 == 0. Weight loads leave no trace in the caches (nontemporal): a model's weights are gone
// from them before its next step (5 rows, 2048 x 2048: 4.7 us, 5.0 through the caches). Weights of
// a model that the last-level cache could hold pay for it (16 rows, 1024 x 4096: 7.7 and 6.2).
//
// One launch can take several weights of the same input (q, k and v; gate and
// up), each with an output of its own, and can return silu(gate) * up instead of
// gate and up; one weight can also be split into groups of rows that take
// different inputs. A launch of a small weight alone does not reach the memory's
// rate: 1024 x 4096 takes 5 us, 1.7 us of them for its bytes.

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <climits>
#include <type_traits>

#include "common.h"
#include "gemm_stream.h"
#include "ops_api.h"

namespace amd_ops {

__device__ __forceinline__ float dot2(const bf16x8& a, const bf16x8& b, int j, float c) {
  const gemv_bf16x8 av = __builtin_bit_cast(gemv_bf16x8, a), bv = __builtin_bit_cast(gemv_bf16x8, b);
  return __builtin_amdgcn_fdot2_f32_bf16(gemv_bf16x2{av[2 * j], av[2 * j + 1]},
                                         gemv_bf16x2{bv[2 * j], bv[2 * j + 1]}, c, false);
}

__device__ __forceinline__ bf16x8 load_stream(const bf16* p) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(bf16x8, __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p)));
}

// A wave takes R rows of W, or with GLU one row of gate and the same of up, and
// has 512 U columns of each in flight. One row and U = 8 reach the highest rate
// for one row of x: 14336 x 4096 in 18.6 us (6.3 TB/s) against 23.1 with two rows
// and U = 2, and 24.2 with two rows and U = 1; short rows end before 8 are in flight.
// With two rows of x the loads of x count: two rows of W share them, and in steps of 512
// columns (10240 x 8192 30.5 us, one row in steps of 2048 36.7; 5120 x 17408 32.2 and 39.3;
// 28672 x 3072 0.95 of one row's). Not up to 4096 rows, which leave too few waves (2048 x
// 14336 21.7 and 14.4, 3072 x 8192 14.3 and 11.6), nor for rows of 2048 or 4096 columns,
// which the longer steps divide, below some 128 MB (11008 x 4096 20.0 and 19.0, 12288 x 2048
// 11.6 and 11.1; but 28672 x 4096 41.4 and 43.5, 65536 x 2048 44.1 and 46.0). Weights of
// less than 24 MB keep one row.
template <int B, int R, int U, bool GLU>
__global__ __launch_bounds__(256) void gemv_bf16_kernel(const Rows p) {
  static_assert(!GLU || R == 2);
  constexpr int STEP = GLU ? 1 : R;               // rows of output per wave
  const Segment seg = segment_of(p, blockIdx.x);
  const int K = p.K, N = seg.n;
  const int lane = threadIdx.x & (WAVE_SIZE - 1);
  const int row0 = ((blockIdx.x - seg.first) * 4 + threadIdx.x / WAVE_SIZE) * STEP;
  if (row0 >= N) return;
  float acc[R][B];
  const bf16* w[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    w[r] = GLU ? p.w[r] + (long)row0 * K : seg.w + (long)min(row0 + r, N - 1) * K;
#pragma unroll
    for (int b = 0; b < B; ++b) acc[r][b] = 0.f;
  }
  const bf16* x = p.x;
  if (p.group_n) x += (long)(row0 / p.group_n) * B * K;   // group_n is a multiple of R
  auto part = [&](int k, auto depth) {
    constexpr int D = decltype(depth)::value;
    bf16x8 wv[D][R];
#pragma unroll
    for (int u = 0; u < D; ++u)
#pragma unroll
      for (int r = 0; r < R; ++r) wv[u][r] = load_stream(w[r] + k + u * 512);
#pragma unroll
    for (int u = 0; u < D; ++u)
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const bf16x8 xv = *reinterpret_cast<const bf16x8*>(x + (long)b * K + k + u * 512);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          float d = 0.f;
#pragma unroll
          for (int j = 0; j < 4; ++j) d = dot2(wv[u][r], xv, j, d);   // f32 accumulation
          acc[r][b] += d;
        }
      }
  };
  int k = lane * 8;                               // K % 8 == 0: all 8 columns or none
  for (; k + 512 * (U - 1) < K; k += 512 * U) part(k, std::integral_constant<int, U>{});
  if constexpr (U > 4) {
    if (k + 512 * 3 < K) {
      part(k, std::integral_constant<int, 4>{});
      k += 512 * 4;
    }
  }
  for (; k < K; k += 512) part(k, std::integral_constant<int, 1>{});
#pragma unroll
  for (int b = 0; b < B; ++b) {
    float t[R];
#pragma unroll
    for (int r = 0; r < R; ++r) t[r] = wave_reduce_sum(acc[r][b]);
    if (lane != 0) continue;
    if constexpr (GLU) {
      p.y[0][(long)b * N + row0] = f2bf(silu_mul(t[0], t[1]));
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (row0 + r >= N) break;
        if (p.bias) t[r] += bf2f(p.bias[row0 + r]);
        if (p.relu2) {
          t[r] = fmaxf(t[r], 0.f);
          t[r] *= t[r];
        }
        if (p.res) t[r] += bf2f(p.res[(long)b * N + row0 + r]);
        if (p.yf) p.yf[(long)b * N + row0 + r] = t[r];
        else seg.y[(long)b * N + row0 + r] = f2bf(t[r]);
      }
    }
  }
}

// A workgroup takes 16 RT rows of W (GLU: 16 of gate and the same 16 of up) and
// 16 NB rows of x; its waves take a part of K each and add up through LDS at the
// end, so that N = 1024 fills the chip too. Matrix fragments want one row per lane,
// memory wants consecutive lanes on consecutive bytes: each wave moves its tiles of W
// and x with coalesced loads into LDS of its own, with the next tile's loads in flight
// (two ahead: the same). No workgroup barrier in the loop.
constexpr int SK_KC = 128;                        // K per tile
constexpr int SK_STRIDE = SK_KC * 2 + 16;         // LDS bytes per row

template <int NB, int WAVES, int RT, bool GLU>
__global__ __launch_bounds__(WAVES * WAVE_SIZE) void gemm_skinny_kernel(const Rows p, int B) {
  static_assert(!GLU || RT == 2);
  constexpr int OUT = GLU ? 16 : 16 * RT;         // rows of output per workgroup
  constexpr int RS = 16 * NB + 1;
  constexpr int RED = WAVES * 16 * RT * RS * 4;
  constexpr int TILE = 16 * (RT + NB) * SK_STRIDE;
  __shared__ __attribute__((aligned(16))) char lds[WAVES * TILE > RED ? WAVES * TILE : RED];
  const int lane = threadIdx.x & (WAVE_SIZE - 1), wid = threadIdx.x / WAVE_SIZE;
  const int lo16 = lane & 15, hi4 = lane >> 4;
  const Segment seg = segment_of(p, blockIdx.x);
  const int K = p.K, N = seg.n;
  const int n0 = (blockIdx.x - seg.first) * OUT;
  const bf16* x = p.x;
  if (p.group_n) x += (long)(n0 / p.group_n) * B * K;   // group_n % OUT == 0
  char* wl = lds + wid * TILE;                    // [16 RT][SK_STRIDE]
  char* xl = wl + 16 * RT * SK_STRIDE;            // [16 NB][SK_STRIDE]

  gemv_f32x4 acc[RT][NB];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[r][b] = gemv_f32x4{0.f, 0.f, 0.f, 0.f};
  const int tiles = (K + SK_KC - 1) / SK_KC, per = (tiles + WAVES - 1) / WAVES;
  const int step = p.stretches ? 1 : WAVES;
  const int t_lo = p.stretches ? wid * per : wid, t_hi = p.stretches ? min(t_lo + per, tiles) : tiles;

  // load j covers rows 4j + hi4, 16 bytes per lane at column 8 lo16
  bf16x8 wr[4 * RT], xr[4 * NB];
  auto fetch = [&](int t) {
    const int k = t * SK_KC + lo16 * 8;
    const bool in = k < K;                        // K % 8 == 0: all 8 or none
#pragma unroll
    for (int j = 0; j < 4 * RT; ++j) {
      wr[j] = bf16x8{};
      const bf16* w = GLU ? p.w[j / 4] : seg.w;
      const int row = n0 + 4 * (GLU ? j % 4 : j) + hi4;
      if (in) wr[j] = load_stream(w + (long)min(row, N - 1) * K + k);
    }
#pragma unroll
    for (int j = 0; j < 4 * NB; ++j) {
      xr[j] = bf16x8{};
      if (in)
        xr[j] = *reinterpret_cast<const bf16x8*>(x + (long)min(4 * j + hi4, B - 1) * K + k);
    }
  };
  if (t_lo < t_hi) fetch(t_lo);
  for (int t = t_lo; t < t_hi; t += step) {
#pragma unroll
    for (int j = 0; j < 4 * RT; ++j)
      *reinterpret_cast<bf16x8*>(wl + (4 * j + hi4) * SK_STRIDE + lo16 * 16) = wr[j];
#pragma unroll
    for (int j = 0; j < 4 * NB; ++j)
      *reinterpret_cast<bf16x8*>(xl + (4 * j + hi4) * SK_STRIDE + lo16 * 16) = xr[j];
    __builtin_amdgcn_wave_barrier();
    if (t + step < t_hi) fetch(t + step);
#pragma unroll
    for (int kk = 0; kk < SK_KC / 32; ++kk) {
      const int off = lo16 * SK_STRIDE + kk * 64 + hi4 * 16;
      gemv_bf16x8 xv[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b)
        xv[b] = *reinterpret_cast<const gemv_bf16x8*>(xl + b * 16 * SK_STRIDE + off);
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        const gemv_bf16x8 wv = *reinterpret_cast<const gemv_bf16x8*>(wl + r * 16 * SK_STRIDE + off);
#pragma unroll
        for (int b = 0; b < NB; ++b)
          acc[r][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, xv[b], acc[r][b], 0, 0, 0);
      }
    }
    __builtin_amdgcn_wave_barrier();              // the tile is overwritten next
  }
  __syncthreads();                                // tiles become the reduction buffer
  float* red = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        red[((wid * RT + r) * 16 + hi4 * 4 + i) * RS + b * 16 + lo16] = acc[r][b][i];
  __syncthreads();
  auto total = [&](int row, int col) {
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) t += red[(w * 16 * RT + row) * RS + col];
    return t;
  };
  for (int i = threadIdx.x; i < OUT * 16 * NB; i += WAVES * WAVE_SIZE) {
    const int row = i % OUT, col = i / OUT;
    if (n0 + row >= N || col >= B) continue;
    const long o = (long)col * N + n0 + row;
    float t = total(row, col);
    if constexpr (GLU) t = silu_mul(t, total(16 + row, col));
    if (p.relu2) {
      t = fmaxf(t, 0.f);
      t *= t;
    }
    if (p.res) t += bf2f(p.res[o]);
    if (p.yf) p.yf[o] = t;
    else seg.y[o] = f2bf(t);
  }
}

namespace {

const bf16* data(const at::Tensor& t) { return reinterpret_cast<const bf16*>(t.data_ptr()); }

// Gives each segment its blocks of ``per`` rows of output; -> blocks in all.
int place(Rows& p, int segments, int per) {
  int blocks = 0;
  for (int s = 0; s < MAX_SEGMENTS; ++s) {
    p.first[s] = s < segments ? blocks : INT_MAX;
    if (s < segments) blocks += (p.n[s] + per - 1) / per;
  }
  return blocks;
}

template <int B, int R, int U, bool GLU = false>
void launch_gemv(Rows p, int segments) {
  const int blocks = place(p, segments, 4 * (GLU ? 1 : R));
  gemv_bf16_kernel<B, R, U, GLU>
      <<<dim3(blocks), dim3(256), 0, c10::hip::getCurrentHIPStream()>>>(p);
}

// one or two rows of x
void gemv_rows(const Rows& p, int segments, int B) {
  long rows = 0;
  for (int s = 0; s < segments; ++s) rows += p.n[s];
  if (B == 1 && p.K > 2048) launch_gemv<1, 1, 8>(p, segments);
  else if (B == 1) launch_gemv<1, 1, 4>(p, segments);
  else if (rows > 4096 && rows * p.K >= (p.K == 2048 || p.K == 4096 ? 64l << 20 : 12l << 20))
    launch_gemv<2, 2, 1>(p, segments);
  else launch_gemv<2, 1, 4>(p, segments);
}

template <int NB, int WAVES, int RT, bool GLU = false>
void launch_skinny(const Rows& rows, int segments, int B) {
  Rows p = rows;
  const int blocks = place(p, segments, GLU ? 16 : 16 * RT);
  gemm_skinny_kernel<NB, WAVES, RT, GLU>
      <<<dim3(blocks), dim3(WAVES * WAVE_SIZE), 0, c10::hip::getCurrentHIPStream()>>>(p, B);
}

template <int R, int D, int WAVES, bool GLU>
void launch_stream(const Rows& rows, int segments, int B) {
  Rows p = rows;
  auto go = [&](auto xr) {
    using S = Stream<R, decltype(xr)::value, D, WAVES, GLU>;
    const int blocks = place(p, segments, S::OUT);
    gemm_stream_kernel<R, decltype(xr)::value, D, WAVES, GLU>
        <<<dim3(blocks), dim3(WAVES * WAVE_SIZE), S::SMEM, c10::hip::getCurrentHIPStream()>>>(p, B);
  };
  if (B <= 8) return go(std::integral_constant<int, 8>{});
  go(std::integral_constant<int, 16>{});
}

// Rows of W a workgroup: the least of (rows + x) times the workgroups of the fullest CU, where x
// stands for the loads of x and the workgroup's beginning and end; of more than one a CU, as far as
// the others fill in for it, x counts otherwise and the fullest for 0.7. In us, 8 and 16 rows of
// x, rows x columns of W:
//  * 8 rows of W, one workgroup a CU: 2048 x 4096 5.3 and 6.1, 16 rows 6.2 and 7.1; but its ring has the CU
//    to itself (4224 x 768, 3 a CU: 5.9, 24 rows 3.7), and its waves want a tile each (1232 x 128,
//    16 rows in 4 waves 2.4, 2.5)
//  * 24: 5120 x 4096 8.8 and 9.8, 16 rows 11.0 and 12.5, 32 rows 9.4 and 10.5
//  * 32: 7168 x 14336 32.5 and 35.0, 16 rows 35.0 and 40.2
//  * 40: 10240 x 8192 26.8 and 27.3, 24 rows 27.7 and 30.2, 64 rows 30.3 and 31.7
//  * 56: 28672 x 4096 36.8 and 37.1, 32 rows 37.8 and 39.2
// No multiples of 16 above 16 for rows of a multiple of 16 KB, whose channels they crowd (8192 x 8192,
// 32 rows 25.6 and 26.0, 16 rows 21.5 and 23.8); nor many rows where rows of W are short, which leaves
// too few waves (28672 x 1024, 16 rows 11.1 and 12.5, 64 rows 12.0 and 12.6; 12032 x 1280, 9 rows of x:
// 48 rows 8.4, 24 rows 7.4).
// The ring: 8 waves where one workgroup has the CU to itself and rows are long (4096 x 4096 7.3 us,
// 4 waves 7.8; 4096 x 2048 6.2, 4 waves 4.9), else 4; two slots, one from 48 rows (gate and up
// of 14336 x 4096, 56 rows and 16 of x: 36.3 us, two slots 37.3), and of more than one workgroup a CU also
// where that lets them share it: 40 rows (28864 x 3072 33.4 us, one slot 31.6; 50352 x 2560, 16 rows of
// x: 48.9 and 43.5), 24 and 32 of short rows (16384 x 512, 9 rows of x: 32 rows in one slot 5.2, in two 6.4), 32
// with many workgroups (28672 x 4096, 16 rows of x: 39.2 and 42.8).
// Against the kernel above, of 1850 shapes and numbers of rows, 128 x 128 to 151936 x 1024 and more columns, one
// or several weights: 0.86 of its time in the mean, in 14 more than 1.03, 1.06 at most.
struct StreamShape {
  int rows, slots, waves;
};

StreamShape stream_shape(const int* n, int segments, int K, int B, bool glu, int group_n) {
  constexpr int CUS = 256;
  const int x = B <= 8 ? 6 : 8, x_more = B <= 8 ? 4 : 12;
  int best = 0;
  bool alone = true, many = false;
  float least = 0.f;
  for (int r : {8, 16, 24, 32, 40, 48, 56, 64}) {
    const int out = glu ? r / 2 : r;
    if (r > 16 && (group_n % out != 0 || (K % 8192 == 0 && r % 16 == 0))) continue;
    if (r > 32 && K <= (B <= 8 ? 2048 : 1536)) continue;
    long blocks = 0;
    for (int s = 0; s < segments; ++s) blocks += (n[s] + out - 1) / out;
    const long full = (blocks + CUS - 1) / CUS;
    if (r == 8 && (full > 1 || K <= 512)) continue;
    float cost = (float)full * (r + x);
    if (full > 1) cost = 0.7f * cost + 0.3f * ((float)blocks / CUS) * (r + x_more);
    if (best && cost >= least) continue;
    best = r;
    least = cost;
    alone = full == 1;
    many = full > 2;
  }
  const bool share = !alone && K <= 2048;
  switch (best) {
    case 8: return {8, 3, 8};
    case 16: return {16, many && K <= 2048 ? 1 : 2, alone && K >= 3072 ? 8 : 4};
    case 24: return {24, share ? 1 : 2, 4};
    case 32: return {32, share || many ? 1 : 2, 4};
    case 40: return {40, alone ? 2 : 1, 4};
    default: return {best, 1, 4};
  }
}

template <bool GLU>
void stream(const Rows& p, int segments, int B) {
  const StreamShape s = stream_shape(p.n, segments, p.K, B, GLU, p.group_n);
  switch (s.rows) {
    case 8: return launch_stream<8, 3, 8, GLU>(p, segments, B);
    case 16:
      if (s.waves == 8) return launch_stream<16, 2, 8, GLU>(p, segments, B);
      if (s.slots == 1) return launch_stream<16, 1, 4, GLU>(p, segments, B);
      return launch_stream<16, 2, 4, GLU>(p, segments, B);
    case 24:
      if (s.slots == 1) return launch_stream<24, 1, 4, GLU>(p, segments, B);
      return launch_stream<24, 2, 4, GLU>(p, segments, B);
    case 32:
      if (s.slots == 1) return launch_stream<32, 1, 4, GLU>(p, segments, B);
      return launch_stream<32, 2, 4, GLU>(p, segments, B);
    case 40:
      if (s.slots == 1) return launch_stream<40, 1, 4, GLU>(p, segments, B);
      return launch_stream<40, 2, 4, GLU>(p, segments, B);
    case 48: return launch_stream<48, 1, 4, GLU>(p, segments, B);
    case 56: return launch_stream<56, 1, 4, GLU>(p, segments, B);
    default: return launch_stream<64, 1, 4, GLU>(p, segments, B);
  }
}

// Workgroups of 16, 32 or 64 rows of W, and 2, 4 or 8 waves in them. What decides is how many
// tiles of 16 rows the fullest CU gets, with the rows of x that each workgroup loads besides;
// a workgroup alone on its CU needs all the waves that fit, several share them. Small K has
// tiles for few waves. Times in us for rows x columns of W, weights from memory:
//  * up to 16 rows of x (K % 128 != 0 or not on 16 bytes): 16 rows of W, 8 waves (4096 x 4096 7.7, 4 waves 9.1; 10240 x 8192 29.6
//    and 34.7), 4 with more workgroups than two a CU and short rows (9216 x 2048 9.2, 8 waves 9.9);
//    32 rows between one and one and a half workgroups a CU (5120 x 5120 12.4, 16 rows 13.5; but
//    8192 x 8192 24.5 and 23.0), and for many rows of x and of W (16 rows, 32000 x 2048 22.8 and 24.8).
//  * up to 32: 32 rows of W where that gives the fullest CU no more (24 rows, 8192 x 8192 26.6 and
//    31.5; 21504 x 4096 36.2 and 40.7), else 16 (9216 x 2048 12.5, 32 rows 14.1); 64 for long rows,
//    many rows of x and a workgroup a CU (32 rows, 9216 x 5120 30.0 and 31.7, 9216 x 8192 43.1 and 46.0).
//  * up to 64: the least sum of tiles and 2/5 (long rows: 3/5) of one a workgroup, out of 16, 32 and
//    64 rows (48 rows, 9216 x 2048 17.8, 32 rows 19.4; 8192 x 8192 40.6, 16 rows 50.1; 10240 x 8192
//    55.4, 16 rows 61.0; 32000 x 2048 35.2, 32 rows 41.5).
//
// Waves of this kernel read neighbouring tiles of K, or a stretch of K each where rows of W lie a multiple of
// 4 KB apart (8 rows of x, neighbours and stretches: 4096 x 2048 6.6 and 6.0 us, 6144 x 4096
// 13.0 and 11.1, 6144 x 8192 22.6 and 19.0; but 4096 x 2560 0.97 to 1, 22016 x 5120 the same).
// Not with more than 4096 columns where a wave's tile has 32 rows of W or more than 32 rows of x
// (gated, 4096 x 8192 22.1 and 23.3; 64 rows of x, 14336 x 8192 0.92 to 1), nor for few workgroups
// and more than 16 rows of x (24 rows, 2048 x 4096 8.7 and 9.4).
void skinny(Rows p, int segments, int B, bool glu) {
  long n = 0;
  for (int s = 0; s < segments; ++s) n += p.n[s];
  bool streams = B <= 16 && p.K % 128 == 0 && p.K < 1 << 25 && (uintptr_t)p.x % 16 == 0;
  for (int s = 0; s < (glu ? 2 : segments); ++s) streams &= (uintptr_t)p.w[s] % 16 == 0;
  if (streams) return glu ? stream<true>(p, segments, B) : stream<false>(p, segments, B);
  p.stretches = p.K % 2048 == 0 && (p.K <= 4096 || !(glu || B > 32)) &&
                (p.K <= 2048 || n > 3072 || B <= 16 || glu);
  if (glu) {
    if (B <= 16) launch_skinny<1, 4, 2, true>(p, segments, B);
    else if (B <= 32) launch_skinny<2, 4, 2, true>(p, segments, B);
    else launch_skinny<4, 2, 2, true>(p, segments, B);
    return;
  }
  constexpr int CUS = 256;
  auto workgroups = [&](int rt) {
    int n = 0;
    for (int s = 0; s < segments; ++s) n += (p.n[s] + 16 * rt - 1) / (16 * rt);
    return n;
  };
  auto fullest = [&](int rt) { return (workgroups(rt) + CUS - 1) / CUS; };
  auto may = [&](int rt) { return p.group_n % (16 * rt) == 0; };
  const int n1 = workgroups(1);
  if (B <= 16) {
    const bool pairs = may(2) && ((n1 > CUS && n1 <= CUS * 3 / 2) || (B > 8 && n1 >= CUS * 7 / 2));
    const bool few = p.K <= 512 || (n1 > 2 * CUS && p.K < 4096);
    if (pairs && n1 > 2 * CUS) launch_skinny<1, 4, 2>(p, segments, B);
    else if (pairs) launch_skinny<1, 8, 2>(p, segments, B);
    else if (few) launch_skinny<1, 4, 1>(p, segments, B);
    else launch_skinny<1, 8, 1>(p, segments, B);
  } else if (B <= 32) {
    const bool pairs = may(2) && 2 * fullest(2) <= fullest(1);
    if (pairs && fullest(2) > 1) launch_skinny<2, 4, 2>(p, segments, B);
    else if (pairs) launch_skinny<2, 8, 2>(p, segments, B);
    else if (may(4) && B > 24 && p.K > 4096 && n1 > 2 * CUS && fullest(4) == 1)
      launch_skinny<2, 4, 4>(p, segments, B);
    else if (n1 > CUS || p.K <= 512) launch_skinny<2, 4, 1>(p, segments, B);
    else launch_skinny<2, 8, 1>(p, segments, B);
  } else {
    const int x = p.K > 2048 ? 3 : 2;              // fifths of a tile
    int best = 1;
    for (int rt : {2, 4})
      if (may(rt) && fullest(rt) * (5 * rt + x) < fullest(best) * (5 * best + x)) best = rt;
    const bool alone = fullest(best) == 1;
    if (best == 4 && alone) launch_skinny<4, 4, 4>(p, segments, B);
    else if (best == 4) launch_skinny<4, 2, 4>(p, segments, B);
    else if (best == 2 && alone) launch_skinny<4, 4, 2>(p, segments, B);
    else if (best == 2) launch_skinny<4, 2, 2>(p, segments, B);
    else if (alone) launch_skinny<4, 4, 1>(p, segments, B);
    else launch_skinny<4, 2, 1>(p, segments, B);
  }
}

// One weight, [B, K] per group of its rows -> (its part of a launch, output).
std::pair<Rows, at::Tensor> single(const char* name, const at::Tensor& x, const at::Tensor& w,
                                   bool relu2, bool out_f32, int64_t group_n, int unit,
                                   int& B) {
  TORCH_CHECK(x.is_cuda() && w.is_cuda() && x.dtype() == at::kBFloat16 &&
                  w.dtype() == at::kBFloat16 && x.dim() == 2 && w.dim() == 2,
              name, ": x [B,K], w [N,K] bf16 on the GPU");
  const int K = (int)x.size(1), N = (int)w.size(0);
  const int groups = group_n > 0 ? (int)((N + group_n - 1) / group_n) : 1;
  TORCH_CHECK(group_n >= 0 && group_n % unit == 0 && x.size(0) % groups == 0, name,
              ": group_n in multiples of ", unit, ", and one [B,K] input per group");
  TORCH_CHECK(w.size(1) == K && K % 8 == 0 && K >= 8 && N >= 1, name, ": K % 8 == 0");
  B = (int)x.size(0) / groups;
  auto y = at::empty({B, N}, x.options().dtype(out_f32 ? at::kFloat : at::kBFloat16));
  Rows p{};
  p.x = data(x);
  p.w[0] = data(w);
  p.n[0] = N;
  if (out_f32) p.yf = y.data_ptr<float>();
  else p.y[0] = reinterpret_cast<bf16*>(y.data_ptr());
  p.relu2 = relu2;
  p.K = K;
  p.group_n = (int)group_n;
  return {p, y};
}

}  // namespace

// which streamed kernel a call of these sizes takes, for the tests
std::tuple<int64_t, int64_t, int64_t> decode_rows_shape(at::IntArrayRef n, int64_t K, int64_t B, bool glu,
                                                        int64_t group_n) {
  TORCH_CHECK(n.size() >= 1 && n.size() <= MAX_SEGMENTS && B >= 3 && B <= 16 && K >= 128 && K % 128 == 0 &&
                  K < 1 << 25 && group_n >= 0 && group_n % 16 == 0,
              "decode_rows_shape: 1 to 3 weights, 3 to 16 rows, K in 128s");
  int sizes[MAX_SEGMENTS] = {};
  for (size_t s = 0; s < n.size(); ++s) {
    TORCH_CHECK(n[s] >= 1 && n[s] < INT_MAX / 2, "decode_rows_shape: rows of a weight");
    sizes[s] = (int)n[s];
  }
  const StreamShape s = stream_shape(sizes, (int)n.size(), (int)K, (int)B, glu, (int)group_n);
  return {s.rows, s.slots, s.waves};
}

// group_n > 0: x holds several [B, K] inputs one after another, and every
// group_n rows of w take the next one.
at::Tensor gemv_bf16(const at::Tensor& x, const at::Tensor& w,
                     const c10::optional<at::Tensor>& bias, bool relu2, bool out_f32,
                     int64_t group_n) {
  const auto xc = x.contiguous(), wc = w.contiguous();
  at::Tensor bc;
  int B = 0;
  auto [p, y] = single("gemv_bf16", xc, wc, relu2, out_f32, group_n, 2, B);
  TORCH_CHECK(B >= 1 && B <= 16, "gemv_bf16: B in [1,16], got ", B,
              " (larger batches belong on hipBLASLt)");
  if (bias.has_value()) {
    TORCH_CHECK(bias->numel() == p.n[0] && bias->dtype() == at::kBFloat16, "bias [N] bf16");
    bc = bias->contiguous();
    p.bias = data(bc);
  }
  switch (B) {
    case 1:
    case 2: gemv_rows(p, 1, B); break;
    case 3: launch_gemv<3, 2, 1>(p, 1); break;
    case 4: launch_gemv<4, 2, 1>(p, 1); break;
    case 8: launch_gemv<8, 2, 1>(p, 1); break;
    case 16: launch_gemv<16, 2, 1>(p, 1); break;
    default: TORCH_CHECK(false, "gemv_bf16: pad B to one of 1,2,3,4,8,16 (python wrapper does)");
  }
  HIP_CHECK_KERNEL();
  return y;
}

at::Tensor gemm_skinny_bf16(const at::Tensor& x, const at::Tensor& w, bool relu2, bool out_f32,
                            int64_t group_n) {
  const auto xc = x.contiguous(), wc = w.contiguous();
  int B = 0;
  auto [p, y] = single("gemm_skinny_bf16", xc, wc, relu2, out_f32, group_n, 16, B);
  TORCH_CHECK(B >= 1 && B <= 64, "gemm_skinny_bf16: 1..64 rows, got ", B);
  skinny(p, 1, B, false);
  HIP_CHECK_KERNEL();
  return y;
}

// x [B, K] against up to three weights [n, K] in one launch -> [B, n] each; glu:
// against gate and up -> silu(x gate^T) * (x up^T) alone. relu2: max(y, 0)^2;
// residual [B, n] of a single weight: added.
std::vector<at::Tensor> decode_rows(const at::Tensor& x, at::TensorList ws, bool glu, bool relu2,
                                    const std::optional<at::Tensor>& residual) {
  const int64_t B = x.size(0), K = x.size(-1);
  TORCH_CHECK(x.is_cuda() && x.dtype() == at::kBFloat16 && x.dim() == 2 && x.is_contiguous() &&
                  B >= 1 && B <= 64 && K >= 8 && K % 8 == 0,
              "decode_rows: x [1..64, K] bf16, K % 8 == 0");
  TORCH_CHECK(ws.size() >= 1 && ws.size() <= MAX_SEGMENTS, "decode_rows: 1 to 3 weights");
  TORCH_CHECK(!glu || (ws.size() == 2 && ws[0].sizes() == ws[1].sizes() && !relu2 && !residual),
              "decode_rows: gate and up of one shape, and nothing after their product");
  Rows p{};
  p.x = data(x);
  p.K = (int)K;
  std::vector<at::Tensor> out;
  for (size_t s = 0; s < ws.size(); ++s) {
    const auto& w = ws[s];
    TORCH_CHECK(w.device() == x.device() && w.dtype() == at::kBFloat16 && w.dim() == 2 &&
                    w.is_contiguous() && w.size(1) == K && w.size(0) >= 1 &&
                    w.size(0) < INT_MAX / 2,
                "decode_rows: weights [n, K] bf16, rows one after another");
    p.w[s] = data(w);
    p.n[s] = (int)w.size(0);
    if (glu && s == 1) break;
    out.push_back(at::empty({B, w.size(0)}, x.options()));
    p.y[s] = reinterpret_cast<bf16*>(out.back().data_ptr());
  }
  const int segments = (int)out.size();
  p.relu2 = relu2;
  if (residual) {
    TORCH_CHECK(segments == 1 && residual->device() == x.device() &&
                    residual->dtype() == at::kBFloat16 && residual->is_contiguous() &&
                    residual->sizes() == out[0].sizes(),
                "decode_rows: residual as the one output");
    p.res = data(*residual);
  }
  if (B > 2) skinny(p, segments, (int)B, glu);
  else if (B == 1 && glu) launch_gemv<1, 2, 4, true>(p, 1);
  else if (glu && B == 2) launch_gemv<2, 2, 4, true>(p, 1);
  else gemv_rows(p, segments, (int)B);
  HIP_CHECK_KERNEL();
  return out;
}

}  // namespace amd_ops
