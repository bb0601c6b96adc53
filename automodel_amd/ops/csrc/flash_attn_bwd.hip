// Flash attention backward (CDNA4, gfx950): deterministic dK/dV (kv-parallel) and dQ
// (q-parallel) kernels of the forward in flash_attn.hip, plus the MFMA and transpose-read
// layout probes.
//
// Both kernels recompute the scores (7 products instead of the 5 of a fused kernel, which
// would have to add dQ with atomics: gradients here are the same bits in every run).
//   bwd_stats: -rowsum(dO * O) and the row's log-sum-exp in units of log2
//   bwd_dkv:   a wave holds 32 K/V rows and their gradients; Q and dO pass by in tiles of
//              64 rows, for all query heads of the group. S[q][k] and dP[q][k] have the
//              key as the accumulator's column, so P and dS are operands of
//              dV^T += dO^T P and dK^T += Q^T dS as they lie (flash_tile.h).
//   bwd_dq:    a wave holds 32 Q/dO rows; K and V pass by; dQ^T += K^T dS^T.
// Tiles come by direct LDS loads into three buffers with one barrier a tile. The loop is
// pipelined over half tiles: while the vector unit turns scores into P and dS, the matrix
// core forms the scores of the next half tile and adds the products of the previous one
// (PIPE; three tiles of head dim 192/192 or 256 do not fit LDS: there two buffers, and the
// phases follow one another).
// For values of 128 columns dK/dV, and dQ of long walks, have kernels of their own with their
// instructions in a given order (flash_dkv.h, flash_dq.h). The others' dK/dV is bound by waits that
// nothing fills: its accumulators and operands leave one wave a SIMD. dQ here, two waves a SIMD, is
// bound by the matrix cores and LDS reads (32 rows per wave: 128 B/clk at full MFMA rate).
// Measured, dK/dV + dQ + stats (causal, bf16, before -> now): 1 x 16384, 32/8 heads of 128:
// 8.04 -> 5.80 ms (dK/dV 5.45 -> 3.75, dQ 2.76 -> 2.3); 2 x 4096: 1069 -> 801 us; 2 x 3001, 16 heads
// (192, 128): 457 -> 320 us; 4 x 2048, 16/8 heads of 64: 176 us; 2 x 4096, 16/8 heads of 256: 1.35 ms.

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <climits>
#include <cmath>

#include "common.h"
#include "flash_tile.h"
#include "ops_api.h"

namespace amd_ops {

using namespace fa;

// stats[0][b][h][s] = lse * log2(e), stats[1][b][h][s] = -rowsum(dO * O), rows padded to
// sp = a multiple of 64; padding rows get a log-sum-exp whose probabilities are 0. A block
// takes 64 rows of one head: 16-byte loads, DV / 8 lanes a row, coalesced stores.
template <int DV>
__global__ __launch_bounds__(256) void bwd_stats_kernel(const bf16* __restrict__ dout,
                                                        const bf16* __restrict__ o,
                                                        const float* __restrict__ lse,
                                                        float* __restrict__ stats, int Sq, int sp,
                                                        int Hq, long plane) {
  constexpr int LANES = DV <= 64 ? 8 : DV <= 128 ? 16 : 32, ROWS = 256 / LANES;
  __shared__ float sum[64];
  const int h = blockIdx.y, b = blockIdx.z, s0 = blockIdx.x * 64;
  const int l = threadIdx.x % LANES;
#pragma unroll
  for (int i = threadIdx.x / LANES; i < 64; i += ROWS) {
    float acc = 0.f;
    if (s0 + i < Sq && l < DV / 8) {
      const long at = (((long)b * Sq + s0 + i) * Hq + h) * DV + l * 8;
      const bf16x8 x = *reinterpret_cast<const bf16x8*>(dout + at);
      const bf16x8 y = *reinterpret_cast<const bf16x8*>(o + at);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc = fmaf(bf2f(x.v[j]), bf2f(y.v[j]), acc);
    }
#pragma unroll
    for (int off = LANES / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if (l == 0) sum[i] = acc;
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const int s = s0 + threadIdx.x;
    const long at = ((long)b * Hq + h) * sp + s;
    stats[at] = s < Sq ? lse[((long)b * Hq + h) * Sq + s] * LOG2E : 1e30f;
    stats[plane + at] = -sum[threadIdx.x];
  }
}

struct BwdArgs {
  const bf16 *dout, *q, *k, *v;
  const float* stats;              // two planes of B * Hq * sp
  bf16 *dq, *dk, *dv;
  float *dk_part, *dv_part;        // [parts][B, Skv, Hk, columns], if a walk is cut into several
  float* dq_part;                  // [q_parts][B, Sq, Hq, columns]
  const int *doc_start, *doc_end;
  int B, Sq, Skv, Hq, Hk, q_start, sp, docs, parts, q_parts;
  long plane;
  float scale;
  bool causal;
};

}  // namespace amd_ops

#include "flash_dkv.h"
#include "flash_dq.h"

namespace amd_ops {

using namespace fa;

template <int D>
__device__ __forceinline__ void load_row_frags(bf16x8_t (&f)[D / 16], const bf16* row) {
  const int half = (threadIdx.x >> 5) & 1;
#pragma unroll
  for (int c = 0; c < D / 16; ++c)
    f[c] = *reinterpret_cast<const bf16x8_t*>(row + c * 16 + half * 8);
}

// ------------------------------------------------------------------------------- dK, dV
template <int DQK, int DV, bool PIPE>
struct Dkv {
  static constexpr int QT = 64 * row_bytes(DQK), OT = 64 * row_bytes(DV), ST = 1024;
  static constexpr int BUF = QT + OT + ST, NBUF = PIPE ? 3 : 2, SMEM = NBUF * BUF;
  char* smem;
  unsigned qrow, orow, qcol, ocol;
  float c;
  bf16x8_t kf[DQK / 16], vf[DV / 16];
  f32x16_t dk[DQK / 32], dv[DV / 32];
  int kpos, kend;
  bool causal;

  // S and dP - delta of the 32 rows `sub` of the tile at byte `buf`
  __device__ __forceinline__ void scores(f32x16_t& s, f32x16_t& dp, unsigned buf, int sub) {
    const int half = (threadIdx.x >> 5) & 1;
    const float* nd = reinterpret_cast<const float*>(smem + buf + QT + OT + 256) + sub * 32 + 4 * half;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float4 w = *reinterpret_cast<const float4*>(nd + 8 * g);
      dp[4 * g] = w.x; dp[4 * g + 1] = w.y; dp[4 * g + 2] = w.z; dp[4 * g + 3] = w.w;
    }
    s = zero16();
#pragma unroll
    for (int ch = 0; ch < DQK / 16; ++ch) s = mma(read_rows<DQK>(smem, buf, qrow, sub, ch), kf[ch], s);
#pragma unroll
    for (int ch = 0; ch < DV / 16; ++ch) dp = mma(read_rows<DV>(smem, buf + QT, orow, sub, ch), vf[ch], dp);
  }

  __device__ __forceinline__ void grads(const bf16x8_t (&p)[2], const bf16x8_t (&ds)[2], unsigned buf,
                                        int sub) {
#pragma unroll
    for (int t = 0; t < DV / 32; ++t)
#pragma unroll
      for (int ch = 0; ch < 2; ++ch)
        dv[t] = mma(read_cols<DV>(smem, buf + QT, ocol, sub, ch, t), p[ch], dv[t]);
#pragma unroll
    for (int t = 0; t < DQK / 32; ++t)
#pragma unroll
      for (int ch = 0; ch < 2; ++ch)
        dk[t] = mma(read_cols<DQK>(smem, buf, qcol, sub, ch, t), ds[ch], dk[t]);
  }

  // scores of 32 rows at position q0.. become the operands P and dS
  template <bool MASK, bool VARLEN>
  __device__ __forceinline__ void probs(f32x16_t& s, f32x16_t& dp, unsigned buf, int sub, int q0,
                                        bf16x8_t (&p)[2], bf16x8_t (&ds)[2]) {
    const int half = (threadIdx.x >> 5) & 1;
    const float* l2 = reinterpret_cast<const float*>(smem + buf + QT + OT) + sub * 32 + 4 * half;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float4 w = *reinterpret_cast<const float4*>(l2 + 8 * g);
      const float l[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = 4 * g + j, q = q0 + acc_row(r, half);
        float e = __builtin_amdgcn_exp2f(fmaf(s[r], c, -l[j]));
        if (MASK && ((causal && kpos > q) || (VARLEN && q >= kend))) e = 0.f;
        s[r] = e;
        dp[r] *= e;
      }
    }
    p[0] = pack8(s, 0); p[1] = pack8(s, 1);
    ds[0] = pack8(dp, 0); ds[1] = pack8(dp, 1);
  }
};

// a lane's row of sums, as the accumulators have it
template <int D>
__device__ __forceinline__ void keep_row(const f32x16_t (&acc)[D / 32], float* row) {
  const int half = (threadIdx.x >> 5) & 1;
#pragma unroll
  for (int t = 0; t < D / 32; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<float4*>(row + t * 32 + 8 * g + 4 * half) =
          float4{acc[t][4 * g], acc[t][4 * g + 1], acc[t][4 * g + 2], acc[t][4 * g + 3]};
}

// out = bf16(scale * the sum of the parts), in their order; n is a multiple of 8
struct PartSums {
  const float* part;
  bf16* out;
  long n;
  float scale;
  int parts;
};
__global__ __launch_bounds__(256) void add_walks_kernel(const PartSums k, const PartSums v, const PartSums q) {
  long i = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
  const bool first = i < k.n, second = !first && i < k.n + v.n;
  if (!first) i -= k.n;
  if (!first && !second) i -= v.n;
  const PartSums& s = first ? k : second ? v : q;
  if (i >= s.n) return;
  float4 lo = *reinterpret_cast<const float4*>(s.part + i), hi = *reinterpret_cast<const float4*>(s.part + i + 4);
  for (int p = 1; p < s.parts; ++p) {
    const float4 x = *reinterpret_cast<const float4*>(s.part + p * s.n + i);
    const float4 y = *reinterpret_cast<const float4*>(s.part + p * s.n + i + 4);
    lo.x += x.x; lo.y += x.y; lo.z += x.z; lo.w += x.w;
    hi.x += y.x; hi.y += y.y; hi.z += y.z; hi.w += y.w;
  }
  bf16x8 o;
  const float f[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
  for (int e = 0; e < 8; ++e) o.v[e] = f2bf(f[e] * s.scale);
  *reinterpret_cast<bf16x8*>(s.out + i) = o;
}

template <int DQK, int DV, int WAVES, int OCC, bool PIPE, bool VARLEN>
__global__ __launch_bounds__(64 * WAVES, OCC) void bwd_dkv_kernel(const BwdArgs a) {
  using F = Dkv<DQK, DV, PIPE>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int BM = WAVES * 32;
  F f;
  f.smem = smem;
  f.qrow = rows_base<DQK>(); f.orow = rows_base<DV>();
  f.qcol = cols_base<DQK>(); f.ocol = cols_base<DV>();
  f.c = a.scale * LOG2E;
  f.causal = a.causal;

  const Place at = place_block((a.Skv + BM - 1) / BM, a.Hk * a.parts, a.B, false);
  const int lane = threadIdx.x & 63, col = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kvh = at.head / a.parts, part = at.head % a.parts, b = at.batch, G = a.Hq / a.Hk;
  const int kvb = at.tile * BM, kv0 = kvb + wid * 32;
  const int row = min(kv0 + col, a.Skv - 1);            // rows beyond Skv are not stored
  load_row_frags<DQK>(f.kf, a.k + (((long)b * a.Skv + row) * a.Hk + kvh) * DQK);
  load_row_frags<DV>(f.vf, a.v + (((long)b * a.Skv + row) * a.Hk + kvh) * DV);
#pragma unroll
  for (int t = 0; t < DQK / 32; ++t) f.dk[t] = zero16();
#pragma unroll
  for (int t = 0; t < DV / 32; ++t) f.dv[t] = zero16();
  f.kpos = kv0 + col;
  f.kend = VARLEN ? a.doc_end[row] : 0;

  // query tiles that see some row of the block, or a part of them, and a wave's first masked positions
  int j0 = a.causal && kvb > a.q_start ? (kvb - a.q_start) / 64 : 0;
  int j1 = (a.Sq + 63) / 64, end_w = 0x7fffffff;
  if (VARLEN) {
    const int de = __builtin_amdgcn_readfirstlane(a.doc_end[min(kvb + BM, a.Skv) - 1]);
    j1 = min(j1, (de - a.q_start + 63) / 64);
    end_w = __builtin_amdgcn_readfirstlane(a.doc_end[min(kv0, a.Skv - 1)]);
  }
  part_of_walk(j0, j1, part, a.parts);
  const int nt = max(j1 - j0, 0), total = nt * G;
  const unsigned q_rs = (unsigned)a.Hq * DQK * 2, o_rs = (unsigned)a.Hq * DV * 2;

  const unsigned lds = lds_address(smem);
  auto load = [&](int u, unsigned buf) {
    const int h = kvh * G + u / nt, q0 = (j0 + u % nt) * 64;
    load_tile<DQK, 64, WAVES>(a.q + (((long)b * a.Sq + q0) * a.Hq + h) * DQK, q_rs, a.Sq - q0,
                              lds + buf);
    load_tile<DV, 64, WAVES>(a.dout + (((long)b * a.Sq + q0) * a.Hq + h) * DV, o_rs, a.Sq - q0,
                             lds + buf + F::QT);
    if (wid == 0) {      // 64 rows of both statistics, 16 bytes a lane (lanes 32.. repeat)
      const float* src = a.stats + ((long)b * a.Hq + h) * a.sp + q0;
      const float* mine = src + (lane & 15) * 4 + ((lane >> 4) & 1) * a.plane;
      load_lds16(lds + buf + F::QT + F::OT, mine);
    }
  };
  auto masked = [&](int u) {
    const int q0 = a.q_start + (j0 + u % nt) * 64;
    return (a.causal && q0 < kv0 + 31) || (VARLEN && q0 + 63 >= end_w);
  };
  auto pos = [&](int u) { return a.q_start + (j0 + u % nt) * 64; };

  if (total > 0) {
    f32x16_t s0, d0;
    bf16x8_t p0[2], e0[2];
    load(0, 0);
    if constexpr (PIPE) {
      f32x16_t s1, d1;
      bf16x8_t p1[2], e1[2];
      if (total > 1) load(1, F::BUF);
      wait_loads();
      barrier();
      f.scores(s0, d0, 0, 0);
      unsigned prev = 0, cur = 0, next = F::BUF, free = 2 * F::BUF;
      for (int u = 0; u < total; ++u) {
        const bool mask = masked(u);
        f.scores(s1, d1, cur, 1);
        if (u > 0) f.grads(p1, e1, prev, 1);
        if (mask) f.template probs<true, VARLEN>(s0, d0, cur, 0, pos(u), p0, e0);
        else f.template probs<false, VARLEN>(s0, d0, cur, 0, pos(u), p0, e0);
        wait_loads();     // the tile u + 1; the buffer of u - 1 is free
        barrier();
        if (u + 2 < total) load(u + 2, free);
        f.scores(s0, d0, next, 0);    // (after the last tile: not used)
        f.grads(p0, e0, cur, 0);
        if (mask) f.template probs<true, VARLEN>(s1, d1, cur, 1, pos(u) + 32, p1, e1);
        else f.template probs<false, VARLEN>(s1, d1, cur, 1, pos(u) + 32, p1, e1);
        prev = cur; cur = next; next = free; free = prev;
      }
      f.grads(p1, e1, prev, 1);
    } else {
      for (int u = 0; u < total; ++u) {
        const unsigned buf = (u & 1) * F::BUF;
        const bool mask = masked(u);
        wait_loads();     // the tile u; the other buffer is free
        barrier();
        if (u + 1 < total) load(u + 1, F::BUF - buf);
#pragma unroll 1
        for (int sub = 0; sub < 2; ++sub) {
          f.scores(s0, d0, buf, sub);
          if (mask) f.template probs<true, VARLEN>(s0, d0, buf, sub, pos(u) + 32 * sub, p0, e0);
          else f.template probs<false, VARLEN>(s0, d0, buf, sub, pos(u) + 32 * sub, p0, e0);
          f.grads(p0, e0, buf, sub);
        }
      }
    }
    barrier();
  }
  if (a.parts > 1) {           // sums in 32 bits, which are added up later
    if (kv0 + col < a.Skv) {
      const long at_row = (((long)part * a.B + b) * a.Skv + kv0 + col) * a.Hk + kvh;
      keep_row<DQK>(f.dk, a.dk_part + at_row * DQK);
      keep_row<DV>(f.dv, a.dv_part + at_row * DV);
    }
    return;
  }
  char* mine = smem + wid * 32 * row_bytes(DQK > DV ? DQK : DV);
  const long first = ((long)b * a.Skv + kv0) * a.Hk + kvh;
  store_rows<DQK>(f.dk, a.scale, mine, a.dk + first * DQK, (long)a.Hk * DQK, a.Skv - kv0);
  store_rows<DV>(f.dv, 1.f, mine, a.dv + first * DV, (long)a.Hk * DV, a.Skv - kv0);
}

// ----------------------------------------------------------------------------------- dQ
template <int DQK, int DV, bool PIPE>
struct Dq {
  static constexpr int KT = 64 * row_bytes(DQK), VT = 64 * row_bytes(DV);
  static constexpr int NK = PIPE ? 3 : 2, SMEM = NK * KT + 2 * VT;   // K is read once more, later
  char* smem;
  unsigned krow, vrow, kcol;
  float c, l2, nd;
  bf16x8_t qf[DQK / 16], of[DV / 16];
  f32x16_t dq[DQK / 32];
  int qpos, qdoc, skv;
  bool causal;

  __device__ __forceinline__ void scores(f32x16_t& s, f32x16_t& dp, unsigned kt, unsigned vt, int sub) {
    s = zero16();
#pragma unroll
    for (int r = 0; r < 16; ++r) dp[r] = nd;
#pragma unroll
    for (int ch = 0; ch < DQK / 16; ++ch) s = mma(read_rows<DQK>(smem, kt, krow, sub, ch), qf[ch], s);
#pragma unroll
    for (int ch = 0; ch < DV / 16; ++ch) dp = mma(read_rows<DV>(smem, vt, vrow, sub, ch), of[ch], dp);
  }
  __device__ __forceinline__ void grads(const bf16x8_t (&ds)[2], unsigned kt, int sub) {
#pragma unroll
    for (int t = 0; t < DQK / 32; ++t)
#pragma unroll
      for (int ch = 0; ch < 2; ++ch)
        dq[t] = mma(read_cols<DQK>(smem, kt, kcol, sub, ch, t), ds[ch], dq[t]);
  }
  template <bool MASK, bool VARLEN>
  __device__ __forceinline__ void probs(f32x16_t& s, f32x16_t& dp, int k0, bf16x8_t (&ds)[2]) {
    const int half = (threadIdx.x >> 5) & 1;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int k = k0 + acc_row(r, half);
      float e = __builtin_amdgcn_exp2f(fmaf(s[r], c, -l2));
      if (MASK && ((causal && k > qpos) || k >= skv || (VARLEN && k < qdoc))) e = 0.f;
      dp[r] *= e;
    }
    ds[0] = pack8(dp, 0); ds[1] = pack8(dp, 1);
  }
};

template <int DQK, int DV, int WAVES, int OCC, bool PIPE, bool VARLEN>
__global__ __launch_bounds__(64 * WAVES, OCC) void bwd_dq_kernel(const BwdArgs a) {
  using F = Dq<DQK, DV, PIPE>;
  constexpr int KT = F::KT, VT = F::VT, V0 = F::NK * KT;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int BM = WAVES * 32;
  F f;
  f.smem = smem;
  f.krow = rows_base<DQK>(); f.vrow = rows_base<DV>(); f.kcol = cols_base<DQK>();
  f.c = a.scale * LOG2E;
  f.causal = a.causal;
  f.skv = a.Skv;

  const Place at = place_block((a.Sq + BM - 1) / BM, a.Hq * a.q_parts, a.B, a.causal);
  const int lane = threadIdx.x & 63, col = lane & 31;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = at.head / a.q_parts, part = at.head % a.q_parts, b = at.batch, kvh = h / (a.Hq / a.Hk);
  const int qblk = at.tile * BM, q0 = qblk + wid * 32;
  const int row = min(q0 + col, a.Sq - 1);              // rows beyond Sq are not stored
  const long qo = ((long)b * a.Sq + row) * a.Hq + h;
  load_row_frags<DQK>(f.qf, a.q + qo * DQK);
  load_row_frags<DV>(f.of, a.dout + qo * DV);
  const float* st = a.stats + ((long)b * a.Hq + h) * a.sp + row;
  f.l2 = st[0];
  f.nd = st[a.plane];
#pragma unroll
  for (int t = 0; t < DQK / 32; ++t) f.dq[t] = zero16();
  f.qpos = a.q_start + q0 + col;
  f.qdoc = VARLEN ? a.doc_start[a.q_start + row] : 0;

  const int last = a.q_start + min(qblk + BM, a.Sq) - 1, all = (a.Skv + 63) / 64;
  int t0 = 0, t1 = a.causal ? min(last / 64 + 1, all) : all, doc_w = 0;
  if (VARLEN) {
    t0 = __builtin_amdgcn_readfirstlane(a.doc_start[a.q_start + qblk]) / 64;
    doc_w = __builtin_amdgcn_readfirstlane(a.doc_start[a.q_start + min(q0 + 32, a.Sq) - 1]);
  }
  part_of_walk(t0, t1, part, a.q_parts);
  const int t_diag = a.causal ? (a.q_start + q0 + 1) / 64 : all;
  const unsigned k_rs = (unsigned)a.Hk * DQK * 2, v_rs = (unsigned)a.Hk * DV * 2;
  const bf16* kp = a.k + ((long)b * a.Skv * a.Hk + kvh) * DQK;
  const bf16* vp = a.v + ((long)b * a.Skv * a.Hk + kvh) * DV;
  const unsigned lds = lds_address(smem);
  auto load_k = [&](int t, unsigned to) {
    load_tile<DQK, 64, WAVES>(kp + (long)t * 64 * a.Hk * DQK, k_rs, a.Skv - t * 64, lds + to);
  };
  auto load_v = [&](int t) {
    load_tile<DV, 64, WAVES>(vp + (long)t * 64 * a.Hk * DV, v_rs, a.Skv - t * 64,
                             lds + V0 + (t & 1) * VT);
  };
  auto masked = [&](int t) {
    return t >= t_diag || t * 64 + 64 > a.Skv || (VARLEN && t * 64 < doc_w);
  };

  if (t0 < t1) {
    f32x16_t s0, d0;
    bf16x8_t e0[2];
    load_k(t0, 0);
    load_v(t0);
    if constexpr (PIPE) {
      f32x16_t s1, d1;
      bf16x8_t e1[2];
      wait_loads();
      barrier();
      if (t0 + 1 < t1) { load_k(t0 + 1, KT); load_v(t0 + 1); }
      f.scores(s0, d0, 0, V0 + (t0 & 1) * VT, 0);
      unsigned prev = 0, cur = 0, next = KT, free = 2 * KT;
      for (int t = t0; t < t1; ++t) {
        const bool mask = masked(t);
        const unsigned vt = V0 + (t & 1) * VT, vn = V0 + ((t + 1) & 1) * VT;
        f.scores(s1, d1, cur, vt, 1);
        if (t > t0) f.grads(e1, prev, 1);
        if (mask) f.template probs<true, VARLEN>(s0, d0, t * 64, e0);
        else f.template probs<false, VARLEN>(s0, d0, t * 64, e0);
        wait_loads();     // K and V of t + 1; the buffers of K of t - 1 and V of t are free
        barrier();
        if (t + 2 < t1) { load_k(t + 2, free); load_v(t + 2); }
        f.scores(s0, d0, next, vn, 0);    // (after the last tile: not used)
        f.grads(e0, cur, 0);
        if (mask) f.template probs<true, VARLEN>(s1, d1, t * 64 + 32, e1);
        else f.template probs<false, VARLEN>(s1, d1, t * 64 + 32, e1);
        prev = cur; cur = next; next = free; free = prev;
      }
      f.grads(e1, prev, 1);
    } else {
      for (int t = t0; t < t1; ++t) {
        const bool mask = masked(t);
        const unsigned kt = ((t - t0) & 1) * KT, vt = V0 + (t & 1) * VT;
        wait_loads();     // K and V of t; the other buffers are free
        barrier();
        if (t + 1 < t1) { load_k(t + 1, KT - kt); load_v(t + 1); }
#pragma unroll 1
        for (int sub = 0; sub < 2; ++sub) {
          f.scores(s0, d0, kt, vt, sub);
          if (mask) f.template probs<true, VARLEN>(s0, d0, t * 64 + 32 * sub, e0);
          else f.template probs<false, VARLEN>(s0, d0, t * 64 + 32 * sub, e0);
          f.grads(e0, kt, sub);
        }
      }
    }
    barrier();
  }
  if (a.q_parts > 1) {
    if (q0 + col < a.Sq)
      keep_row<DQK>(f.dq, a.dq_part + ((((long)part * a.B + b) * a.Sq + q0 + col) * a.Hq + h) * DQK);
    return;
  }
  store_rows<DQK>(f.dq, a.scale, smem + wid * 32 * row_bytes(DQK),
                  a.dq + (((long)b * a.Sq + q0) * a.Hq + h) * DQK, (long)a.Hq * DQK, a.Sq - q0);
}

// Which of the two for values of 128 columns. The ordered kernel has half the workgroups, one on a CU,
// and more to do before its first product: it takes long walks, for 128 / 128 enough of them to fill
// the chip. Whole backward, this one over the other: (192, 128): 0.85 at 2 x 3001 x 16 heads, 0.95 at 1024 to
// 4096 x 8 to 16 heads, 1.0 to 1.02 at 512, 1.05 at 200; 128 / 128: 0.92 at 2 x 4096 x 32 heads, 0.96 at
// 2 x 3001 x 16 (384 workgroups), with 256 of them 1.02 causal and 0.94 without a mask (2048 x 32 heads),
// with 128 1.04 (4096 x 8 heads). Packed documents are short walks: dQ of 6001 tokens in 9 of them,
// 16/8 heads: 77 us, 100 with the ordered kernel.
template <int DQK, int DV>
static bool dq_ordered(const BwdArgs& a) {
  const long blocks = (long)((a.Sq + DqTile<DQK, DV>::BM - 1) / DqTile<DQK, DV>::BM) * a.Hq * a.B;
  return !a.doc_start && a.Skv >= 1024 && a.Sq >= DqTile<DQK, DV>::BM && (DQK == 192 || blocks >= (a.causal ? 384 : 256));
}

// The ordered dK/dV of 128 columns, but for walks of a few tiles of queries, where what a workgroup does
// before and after them counts (whole backward, this one over the other, keys 2048 to 4096: 1.09
// and 1.12 at 16 and 64 queries of 8 x 32 heads, 1.04 and 1.07 at 100 of 16 x 16, the same at 192).
// Of packed rows the walk is a document's, on average, times the heads of a group. (128, 128), 8192
// tokens, 32 / 32 heads: 1.04 at 64 and 100 tokens a document, 1.01 at 200, 0.99 at 256, 0.93 at 700; 16384, 16 / 16:
// 1.05, 1.04, 1.01, 0.99, 0.95; 32 / 8 heads: 1.01, 0.99, 0.98, 0.98, 0.99. (192, 128), 8192, 32: 1.03,
// 1.01, 0.98, 0.96, 0.90; 4096, 32: 1.02, 1.02, 0.99, 0.98, 0.91.
template <int DQK>
static bool dkv_ordered(const BwdArgs& a) {
  const long G = a.Hq / a.Hk;
  if (a.doc_end) return a.docs <= 0 || a.Skv * G >= (DQK == 128 ? 256l : 192l) * a.docs;
  return a.Sq * G >= 192;
}

// Into how many parts the walk of a workgroup over the query tiles is cut. With few key heads there are fewer
// workgroups than CUs (2 x 2048, 16/4 heads: 128), and causal ones of unequal walks take as long as the longest
// (1 x 4096, 32/8 heads: 256). A part's sums go to memory in 32 bits and are added after. Time, in us, by what
// a tile takes, how many workgroups a CU has, and the memory's rate: the longest walk or all of them on all
// CUs, 4 tiles' time for a workgroup's beginning and end, and the adding. Of packed rows the lengths are not
// known here: cuts at random have their longest document at about (ln n + 0.6) of the mean, and half their
// tokens lie in documents of twice that. Whole backward, cut over uncut, 198 shapes of 100 to 16000 queries:
// 0.79 in the mean, 0.27 (1 x 2048, 8/2 heads of 256) to 1.0; 48 of packed rows 0.81, 0.33 to
// 1.0. Always the best of 1, 2, 3, 4, 6 and 8 parts would be 1.4% faster.
static int dkv_parts(const BwdArgs& a, int dqk, int dv) {
  if (a.doc_end && a.docs <= 0) return 1;
  const bool two = dqk == 64;                            // workgroups a CU
  const float tile = two ? 3.4f : dqk == 96 ? 2.5f : dv == 128 ? (dqk == 128 ? 1.75f : 2.15f) : dqk == 192 ? 4.2f : 6.9f;
  const long blocks = (a.Skv + 127) / 128, G = a.Hq / a.Hk, heads = (long)a.Hk * a.B, all = (a.Sq + 63) / 64;
  float longest = 0.f, sum = 0.f;                        // tiles, of one head
  if (a.doc_end) {
    const float mean = (float)a.Skv / a.docs;
    longest = std::min<float>(all, a.docs > 1 ? mean * (std::log((float)a.docs) + .58f) / 64 + 1 : all);
    sum = blocks * (mean * a.docs / (a.docs + 1) / 64 + 2);
  } else {
    for (long t = 0; t < blocks; ++t) {
      const long from = a.causal ? std::max<long>(t * 128 - a.q_start, 0) / 64 : 0;
      const float n = std::max<long>(all - from, 0);
      longest = std::max(longest, n);
      sum += n;
    }
  }
  longest *= G;
  sum *= G * heads;
  const float n = blocks * heads, slots = two ? 512 : 256, ends = 4 * tile;
  const float columns = heads * (float)a.Skv * (dqk + dv);
  auto time = [&](int parts) {
    const float one = two && n * parts <= 256 ? .6f * tile : tile;          // alone on its CU
    float t;
    if (a.causal || a.doc_end) t = std::max(longest / parts * one + ends, (sum * tile + n * parts * ends) / slots);
    else t = std::ceil(n * parts / slots) * (longest / parts * one + ends);
    return parts == 1 ? t : t + 8 + columns * (8 * parts + 2) / 6e6f;
  };
  int best = 1;
  float least = .92f * time(1);                          // (it has to be worth it)
  for (const int parts : {2, 3, 4, 6, 8})
    if (parts * G <= longest && time(parts) < least) {
      least = time(parts);
      best = parts;
    }
  return best;
}

// The kernel of dQ, and into how many parts its walks over the key tiles are cut, as dkv_parts: with few heads and
// rows the longest walk is the time (1 x 3001, 4/4 heads: 96 workgroups). Time in us by what a tile takes, alone on its
// CU (of those with two workgroups) or not, the tiles that a workgroup's beginning and end are as long as, and the adding.
// The ordered kernel's workgroups have more rows, so it is cut where the other one is not. Whole backward, cut over uncut,
// 205 shapes of 100 to 16000 queries: 0.97 in the mean, the 44 that are cut 0.85, 0.66 (1 x 3001, 4/4 heads of 128: 130
// and 86 us) to 1.02; always the best of both kernels and 1, 2, 3, 4, 6 and 8 parts would be 0.5% faster. Documents
// are short walks, and are not cut.
struct DqPlan {
  bool ordered;
  int parts;
};
static DqPlan plan_dq(const BwdArgs& a, int dqk, int dv) {
  const bool both = dv == 128 && (dqk == 128 || dqk == 192);
  DqPlan best{both && (dqk == 128 ? dq_ordered<128, 128>(a) : dq_ordered<192, 128>(a)), 1};
  if (a.doc_start) return best;
  auto time = [&](bool ordered, int parts) {
    const bool two = !ordered && dqk <= 128;
    const long rows = !ordered ? 128 : dqk == 128 ? DqTile<128, 128>::BM : DqTile<192, 128>::BM;
    const float tile = ordered ? (dqk == 128 ? 2.8f : 2.1f) : dqk <= 96 ? 2.f : dqk == 128 ? 3.f : both ? 2.4f : 4.f;
    const long blocks = (a.Sq + rows - 1) / rows, all = (a.Skv + 63) / 64;
    float longest = 0.f, sum = 0.f;                        // tiles, of one head
    for (long t = 0; t < blocks; ++t) {
      const long last = a.q_start + std::min<long>((t + 1) * rows, a.Sq) - 1;
      const float n = a.causal ? std::min(last / 64 + 1, all) : all;
      longest = std::max(longest, n);
      sum += n;
    }
    const float heads = (float)a.Hq * a.B, n = blocks * heads * parts, slots = two ? 512 : 256;
    const float one = two && n <= 256 ? .7f * tile : tile, ends = (ordered ? 5 : 4) * tile;
    float us;
    if (a.causal) us = std::max(longest / parts * one + ends, (heads * sum * tile + n * ends) / slots);
    else us = std::ceil(n / slots) * (longest / parts * one + ends);
    return parts == 1 ? us : us + 5 + heads * a.Sq * dqk * (8 * parts + 2) / 6e6f;
  };
  float least = .9f * time(best.ordered, 1);               // (it has to be worth it)
  for (int ordered = 0; ordered <= (both ? 1 : 0); ++ordered)
    for (const int parts : {2, 3, 4, 6, 8}) {
      if (parts * 192 > a.Skv) continue;                  // (three tiles)
      const float us = time(ordered, parts);
      if (us >= least) continue;
      least = us;
      best = {ordered != 0, parts};
    }
  return best;
}

template <int DQK, int DV>
static void launch_dq_ordered(const BwdArgs& a, hipStream_t stream) {
  using T = DqTile<DQK, DV>;
  hipLaunchKernelGGL((bwd_dq_ordered_kernel<DQK, DV, BwdArgs>),
                     dim3((unsigned)((long)((a.Sq + T::BM - 1) / T::BM) * a.Hq * a.B * a.q_parts)), dim3(256), T::SMEM,
                     stream, a);
  HIP_CHECK_KERNEL();
}

template <int DV>
static void launch_stats(const BwdArgs& a, const bf16* o, const float* lse, float* stats,
                         hipStream_t stream) {
  hipLaunchKernelGGL((bwd_stats_kernel<DV>), dim3(a.sp / 64, a.Hq, a.B), dim3(256), 0, stream, a.dout, o,
                     lse, stats, a.Sq, a.sp, a.Hq, a.plane);
  HIP_CHECK_KERNEL();
}

template <int DQK, int DV, int WAVES, int OCC, bool PIPE>
static void launch_dkv(const BwdArgs& a, hipStream_t stream) {
  const long blocks = (long)((a.Skv + WAVES * 32 - 1) / (WAVES * 32)) * a.Hk * a.B * a.parts;
  // (the results leave through the same memory)
  constexpr int smem = std::max(Dkv<DQK, DV, PIPE>::SMEM, WAVES * 32 * row_bytes(DQK > DV ? DQK : DV));
  if (a.doc_end)
    hipLaunchKernelGGL((bwd_dkv_kernel<DQK, DV, WAVES, OCC, PIPE, true>), dim3((unsigned)blocks),
                       dim3(64 * WAVES), smem, stream, a);
  else
    hipLaunchKernelGGL((bwd_dkv_kernel<DQK, DV, WAVES, OCC, PIPE, false>), dim3((unsigned)blocks),
                       dim3(64 * WAVES), smem, stream, a);
  HIP_CHECK_KERNEL();
}

template <int DQK, int DV>
static void launch_dkv_ordered(const BwdArgs& a, hipStream_t stream) {
  const dim3 grid((unsigned)((long)((a.Skv + 127) / 128) * a.Hk * a.B * a.parts));
  if (a.doc_end)
    hipLaunchKernelGGL((bwd_dkv_ordered_kernel<DQK, DV, true, BwdArgs>), grid, dim3(256),
                       (DkvTile<DQK, DV>::SMEM), stream, a);
  else
    hipLaunchKernelGGL((bwd_dkv_ordered_kernel<DQK, DV, false, BwdArgs>), grid, dim3(256),
                       (DkvTile<DQK, DV>::SMEM), stream, a);
  HIP_CHECK_KERNEL();
}

template <int DQK, int DV, int WAVES, int OCC, bool PIPE>
static void launch_dq(const BwdArgs& a, hipStream_t stream) {
  const long blocks = (long)((a.Sq + WAVES * 32 - 1) / (WAVES * 32)) * a.Hq * a.B * a.q_parts;
  constexpr int smem = std::max(Dq<DQK, DV, PIPE>::SMEM, WAVES * 32 * row_bytes(DQK));
  if (a.doc_start)
    hipLaunchKernelGGL((bwd_dq_kernel<DQK, DV, WAVES, OCC, PIPE, true>), dim3((unsigned)blocks),
                       dim3(64 * WAVES), smem, stream, a);
  else
    hipLaunchKernelGGL((bwd_dq_kernel<DQK, DV, WAVES, OCC, PIPE, false>), dim3((unsigned)blocks),
                       dim3(64 * WAVES), smem, stream, a);
  HIP_CHECK_KERNEL();
}

std::tuple<at::Tensor, at::Tensor, at::Tensor> flash_attn_bwd(
    const at::Tensor& dout, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
    const at::Tensor& o, const at::Tensor& lse, double scale, bool causal, int64_t q_start,
    const std::optional<at::Tensor>& doc_start, const std::optional<at::Tensor>& doc_end, int64_t docs) {
  const int B = q.size(0), Sq = q.size(1), Hq = q.size(2), Dqk = q.size(3);
  const int Skv = k.size(1), Hk = k.size(2), Dv = v.size(3);
  TORCH_CHECK(q.is_contiguous() && k.is_contiguous() && v.is_contiguous() && o.is_contiguous() &&
                  dout.is_contiguous() && dout.sizes() == o.sizes() && lse.is_contiguous() &&
                  lse.numel() == (long)B * Hq * Sq && k.size(3) == Dqk && v.size(1) == Skv && v.size(2) == Hk,
              "flash_attn_bwd: contiguous tensors of the forward's shapes");
  const bool varlen = doc_start.has_value();
  TORCH_CHECK(varlen == doc_end.has_value(), "doc_start and doc_end go together");
  if (varlen)
    TORCH_CHECK(doc_start->numel() >= q_start + Sq && doc_end->numel() >= Skv,
                "flash_attn_bwd: doc_start and doc_end for every position");
  auto stream = c10::hip::getCurrentHIPStream().stream();
  auto dq = at::empty_like(q);
  auto dk = at::empty_like(k);
  auto dv = at::empty_like(v);
  BwdArgs a{};
  a.dout = reinterpret_cast<const bf16*>(dout.data_ptr());
  a.q = reinterpret_cast<const bf16*>(q.data_ptr());
  a.k = reinterpret_cast<const bf16*>(k.data_ptr());
  a.v = reinterpret_cast<const bf16*>(v.data_ptr());
  a.dq = reinterpret_cast<bf16*>(dq.data_ptr());
  a.dk = reinterpret_cast<bf16*>(dk.data_ptr());
  a.dv = reinterpret_cast<bf16*>(dv.data_ptr());
  a.doc_start = varlen ? doc_start->data_ptr<int>() : nullptr;
  a.doc_end = varlen ? doc_end->data_ptr<int>() : nullptr;
  a.B = B; a.Sq = Sq; a.Skv = Skv; a.Hq = Hq; a.Hk = Hk; a.q_start = (int)q_start;
  a.sp = (Sq + 63) / 64 * 64;
  a.plane = (long)B * Hq * a.sp;
  a.scale = (float)scale;
  a.causal = causal;
  a.docs = (int)std::min<int64_t>(docs, INT_MAX);
  auto stats = at::empty({2, B, Hq, a.sp}, q.options().dtype(at::kFloat));
  a.stats = stats.data_ptr<float>();
  const bf16* op = reinterpret_cast<const bf16*>(o.data_ptr());

  // Waves per SIMD and pipelining by what fits the registers and LDS; dK/dV need one wave a
  // SIMD from head dim 96 on (at two a SIMD it spills); values of 128 columns have the ordered kernel for
  // all but the shortest walks. dQ of 128/128 at two waves a SIMD overlaps as well without the third
  // K buffer (379 against 392 us); (192, 128) would spill there (461 against 203 us).
  a.parts = dkv_parts(a, Dqk, Dv);
  at::Tensor part, q_part;
  const DqPlan dq_plan = plan_dq(a, Dqk, Dv);
  a.q_parts = dq_plan.parts;
  if (a.q_parts > 1) {
    q_part = at::empty({a.q_parts * q.numel()}, q.options().dtype(at::kFloat));
    a.dq_part = q_part.data_ptr<float>();
  }
  if (a.parts > 1) {
    part = at::empty({a.parts * (k.numel() + v.numel())}, q.options().dtype(at::kFloat));
    a.dk_part = part.data_ptr<float>();
    a.dv_part = a.dk_part + a.parts * k.numel();
  }
  bool done = false;
#define FA_BWD_CASE(A, C, KV_OCC, KV_PIPE, Q_OCC, Q_PIPE)                                 \
  if (!done && Dqk == A && Dv == C) {                                                     \
    done = true;                                                                          \
    launch_stats<C>(a, op, lse.data_ptr<float>(), stats.data_ptr<float>(), stream);       \
    bool ordered = false;                                                                 \
    if constexpr (C == 128) {                                                             \
      ordered = dkv_ordered<A>(a);                                                        \
      if (ordered) launch_dkv_ordered<A, C>(a, stream);                                   \
    }                                                                                     \
    if (!ordered) launch_dkv<A, C, 4, KV_OCC, KV_PIPE>(a, stream);                        \
    ordered = false;                                                                      \
    if constexpr (C == 128) {                                                             \
      ordered = dq_plan.ordered;                                                          \
      if (ordered) launch_dq_ordered<A, C>(a, stream);                                    \
    }                                                                                     \
    if (!ordered) launch_dq<A, C, 4, Q_OCC, Q_PIPE>(a, stream);                           \
  }
  FA_BWD_CASE(64, 64, 2, true, 2, true)
  FA_BWD_CASE(96, 96, 1, true, 2, true)
  FA_BWD_CASE(128, 128, 1, true, 2, false)
  FA_BWD_CASE(192, 128, 1, true, 1, true)
  FA_BWD_CASE(192, 192, 1, false, 1, false)
  FA_BWD_CASE(256, 256, 1, false, 1, false)
#undef FA_BWD_CASE
  TORCH_CHECK(done, "flash_attn_bwd: unsupported head dims (Dqk=", Dqk, ", Dv=", Dv, ")");
  if (a.parts > 1 || a.q_parts > 1) {
    const PartSums sk{a.dk_part, a.dk, a.parts > 1 ? (long)k.numel() : 0, a.scale, a.parts},
        sv{a.dv_part, a.dv, a.parts > 1 ? (long)v.numel() : 0, 1.f, a.parts},
        sq{a.dq_part, a.dq, a.q_parts > 1 ? (long)q.numel() : 0, a.scale, a.q_parts};
    hipLaunchKernelGGL(add_walks_kernel, dim3((unsigned)((sk.n + sv.n + sq.n + 2047) / 2048)), dim3(256), 0, stream, sk,
                       sv, sq);
    HIP_CHECK_KERNEL();
  }
  return {dq, dk, dv};
}

std::tuple<bool, bool> flash_attn_bwd_ordered(int64_t B, int64_t Sq, int64_t Skv, int64_t Hq, int64_t Hk,
                                              int64_t Dqk, int64_t Dv, bool causal, int64_t docs) {
  TORCH_CHECK(std::min({B, Sq, Skv, Hq, Hk}) >= 1 && std::max({B, Sq, Skv, Hq, Hk, docs}) <= INT_MAX && Hq % Hk == 0,
              "flash_attn_bwd_ordered: sizes");
  if (Dv != 128 || (Dqk != 128 && Dqk != 192)) return {false, false};
  const int here = 0;
  BwdArgs a{};
  a.B = (int)B; a.Sq = (int)Sq; a.Skv = (int)Skv; a.Hq = (int)Hq; a.Hk = (int)Hk;
  a.causal = causal;
  if (docs) a.doc_start = a.doc_end = &here;       // (that there are some is all that is asked)
  a.docs = (int)std::max<int64_t>(docs, 0);
  if (Dqk == 128) return {dkv_ordered<128>(a), dq_ordered<128, 128>(a)};
  return {dkv_ordered<192>(a), dq_ordered<192, 128>(a)};
}

// {whether dQ's kernel is the ordered one, its parts}, of rows that are not packed
std::tuple<bool, int64_t> flash_attn_bwd_dq(int64_t B, int64_t Sq, int64_t Skv, int64_t Hq, int64_t Hk, int64_t Dqk,
                                            int64_t Dv, bool causal, int64_t q_start) {
  TORCH_CHECK(std::min({B, Sq, Skv, Hq, Hk}) >= 1 && std::max({B, Sq, Skv, Hq, Hk, q_start}) <= INT_MAX && Hq % Hk == 0,
              "flash_attn_bwd_dq: sizes");
  BwdArgs a{};
  a.B = (int)B; a.Sq = (int)Sq; a.Skv = (int)Skv; a.Hq = (int)Hq; a.Hk = (int)Hk; a.q_start = (int)q_start;
  a.causal = causal;
  const DqPlan p = plan_dq(a, (int)Dqk, (int)Dv);
  return {p.ordered, p.parts};
}

// dkv_parts; docs: 0 for rows that are not packed
int64_t flash_attn_bwd_parts(int64_t B, int64_t Sq, int64_t Skv, int64_t Hq, int64_t Hk, int64_t Dqk, int64_t Dv,
                             bool causal, int64_t q_start, int64_t docs) {
  TORCH_CHECK(std::min({B, Sq, Skv, Hq, Hk}) >= 1 && std::max({B, Sq, Skv, Hq, Hk, q_start, docs}) <= INT_MAX &&
                  Hq % Hk == 0, "flash_attn_bwd_parts: sizes");
  const int here = 0;
  BwdArgs a{};
  a.B = (int)B; a.Sq = (int)Sq; a.Skv = (int)Skv; a.Hq = (int)Hq; a.Hk = (int)Hk; a.q_start = (int)q_start;
  a.causal = causal;
  if (docs) a.doc_start = a.doc_end = &here;       // (that there are some is all that is asked)
  a.docs = (int)std::max<int64_t>(docs, 0);
  return dkv_parts(a, (int)Dqk, (int)Dv);
}

// ---- MFMA layout self-test: d[32,32] = a[32,16] @ b[16,32] via one mfma.
__global__ void mfma_probe_kernel(const bf16* a, const bf16* b, float* d) {
  const int lane = threadIdx.x & 63;
  const int half = lane >> 5;
  bf16x8_t af, bf_;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    af[j] = (__bf16)a[(lane & 31) * 16 + half * 8 + j];   // A[i=l&31][k=8*half+j]
    bf_[j] = (__bf16)b[(half * 8 + j) * 32 + (lane & 31)];  // B[k=8*half+j][j=l&31]
  }
  f32x16_t acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af, bf_, acc, 0, 0, 0);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = (r & 3) + 8 * (r >> 2) + 4 * half;
    d[row * 32 + (lane & 31)] = acc[r];
  }
}

// ---- ds_read_b64_tr_b16 layout probe: fill LDS with a linear pattern and
// dump what each lane receives for reads at stride-8B lane addresses.
// The gather is the hardware's: this shows what the kernels above rely on.
__global__ void tr16_probe_kernel(const bf16* __restrict__ in, float* __restrict__ out,
                                  int n) {
  __shared__ __attribute__((aligned(16))) bf16 lds[2048];
  const int l = threadIdx.x & 63;
  for (int i = threadIdx.x; i < n; i += 64) lds[i] = in[i];
  __syncthreads();
  // two reads cover 1024 B: lanes at 8-B stride (address = LDS base + offset)
  const unsigned base = (unsigned)(unsigned long long)(uintptr_t)(&lds[0]);
  for (int rd = 0; rd < 2; ++rd) {
    unsigned off = base + (unsigned)(l * 8 + rd * 512);
    unsigned long long v;
    asm volatile("ds_read_b64_tr_b16 %0, %1\n\ts_waitcnt lgkmcnt(0)"
                 : "=v"(v) : "v"(off));
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      unsigned short u = (unsigned short)(v >> (16 * j));
      out[(rd * 64 + l) * 4 + j] = bf2f(__builtin_bit_cast(bf16, u));
    }
  }
}

at::Tensor tr16_probe(const at::Tensor& pattern) {
  TORCH_CHECK(pattern.is_cuda() && pattern.scalar_type() == at::kBFloat16 &&
              pattern.numel() <= 2048, "tr16_probe: bf16, <=2048 elems");
  auto out = at::empty({2, 64, 4}, pattern.options().dtype(at::kFloat));
  auto stream = c10::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(tr16_probe_kernel, dim3(1), dim3(64), 0, stream.stream(),
                     reinterpret_cast<const bf16*>(pattern.data_ptr()),
                     out.data_ptr<float>(), (int)pattern.numel());
  HIP_CHECK_KERNEL();
  return out;
}

at::Tensor mfma_probe(const at::Tensor& a, const at::Tensor& b) {
  TORCH_CHECK(a.is_cuda() && a.sizes() == at::IntArrayRef({32, 16}), "a must be [32,16]");
  TORCH_CHECK(b.sizes() == at::IntArrayRef({16, 32}), "b must be [16,32]");
  auto d = at::empty({32, 32}, a.options().dtype(at::kFloat));
  auto stream = c10::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(mfma_probe_kernel, dim3(1), dim3(64), 0, stream.stream(),
                     reinterpret_cast<const bf16*>(a.data_ptr()),
                     reinterpret_cast<const bf16*>(b.data_ptr()), d.data_ptr<float>());
  HIP_CHECK_KERNEL();
  return d;
}

}  // namespace amd_ops
