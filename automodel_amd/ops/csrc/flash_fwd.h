// The flash-attention forward for values of 128 columns, keys of 128 or 192, without documents
// (gfx950); included by flash_attn.hip.
//
// A wave has 16 N rows of Q with their output in AGPRs, so that an operand from LDS serves N
// products; tiles of 64 rows of K and V pass by. Instructions are in a given order, as in
// flash_dq.h. Over half tiles h of 32 keys a step has S(h + 1) = K Q^T, O^T += V^T P(h - 1) and behind
// the MFMAs P(h) from its scores. S[k][q] leaves a lane (q = lane & 15, g = lane >> 4) with keys
// 4 g + 0..3 of 16: two such tiles are the 8 summed indices of an operand of O^T, as they lie.
//
// What bounds it is that one wave issues: each instruction counts. Rows keep the maximum of their first 32
// keys, and no step looks for another; f32 and bf16 hold what is up to 2^32 above it as well as
// what is below. A sum beyond that is noticed at the end of the step, which is then done again with
// the step's own maximum: its keys are still in LDS.
//
// Three buffers of a tile: K is read one tile ahead of V. One barrier a tile, in the middle of its
// first step.
//
// Two waves a SIMD of 32 rows each, in the compiler's order, read twice as much LDS for a product and
// drew more power: 1 x 16384, 32/8 heads of 128: 2020 -> 1843 us with a causal mask, 4000 -> 3524 (1.25
// PFLOP/s) without; 2 x 3001, 16 heads (192, 128): 110 -> 98 and 216 -> 164 us. Looking for the maximum
// of each half tile took 80 us of the 1843 more.
#pragma once

#include "flash_ordered.h"

namespace amd_ops {
namespace fa {

template <int DQK, int DV, int N_>
struct FwdTile {
  static constexpr int N = N_, ROWS = 16 * N, BM = 4 * ROWS;             // rows of a wave, a workgroup
  static constexpr int KR = DQK * 2, VR = DV * 2;                        // bytes of a row
  static constexpr int KT = 64 * KR, VT = 64 * VR, BUF = KT + VT, SMEM = 3 * BUF;
  // fragments of a step: rows of K, columns of V; how many of them have a place
  static constexpr int F1 = DQK / 16, F = F1 + DV / 16, RING = F / 2;
  static_assert(F % 2 == 0 && RING <= F1 && SMEM <= 160 * 1024 && BM * VR <= SMEM, "places, tiles; the result in them");
  static_assert((DQK / 32 + DV / 16) * N * 4 <= 256, "Q and the output in AGPRs");

  // Operations behind the MFMAs, but the last two. By threes: multiply and add of a score, exponential of the
  // one before, sum with the one before that; then the roundings.
  static constexpr int E = 8 * N, EXPS = 3 * (E + 2), OPS = EXPS + E / 2;
};

__device__ __forceinline__ unsigned pair(float a, float b) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, bf16x2_t{(__bf16)a, (__bf16)b});
}

template <int DQK, int DV, int N, class Args>
__global__ __launch_bounds__(256, 1) void flash_fwd_ordered_kernel(const Args a) {
  using T = FwdTile<DQK, DV, N>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int BUF = T::BUF, KT = T::KT, F1 = T::F1, F = T::F, RING = T::RING, SLOTS = F * N;
  const Place at = place_block((a.Sq + T::BM - 1) / T::BM, a.Hq, a.B, a.causal);
  const int lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = at.head, b = at.batch, kvh = h / (a.Hq / a.Hk);
  const int qblk = at.tile * T::BM, q0 = qblk + wid * T::ROWS;
  const float c = a.scale_log2;

  bf16x8_t qf[N][DQK / 32];
#pragma unroll
  for (int t = 0; t < N; ++t) {
    const int row = min(q0 + 16 * t + i16, a.Sq - 1);        // rows beyond Sq are not stored
    const bf16* src = a.q + (((long)b * a.Sq + row) * a.Hq + h) * DQK + g * 8;
#pragma unroll
    for (int s = 0; s < DQK / 32; ++s) {
      uint4 w = *reinterpret_cast<const uint4*>(src + s * 32);
      if (a.negative) {
        w.x ^= 0x80008000u; w.y ^= 0x80008000u; w.z ^= 0x80008000u; w.w ^= 0x80008000u;
      }
      qf[t][s] = __builtin_bit_cast(bf16x8_t, w);
      asm volatile("" : "+a"(qf[t][s]));                     // (and not four registers that are put together)
    }
  }
  const int qpos = a.q_start + q0 + i16;

  // ---- key tiles that some row of the block sees
  const int last = a.q_start + min(qblk + T::BM, a.Sq) - 1, all = (a.Skv + 63) / 64;
  const int t1 = a.causal ? min(last / 64 + 1, all) : all;
  const int t_diag = a.causal ? (a.q_start + q0 + 1) / 64 : all;
  auto masked = [&](int t) { return t >= t_diag || t * 64 + 64 > a.Skv; };

  f32x4_t o[DV / 16][N];
#pragma unroll
  for (int t = 0; t < DV / 16; ++t)
#pragma unroll
    for (int n = 0; n < N; ++n) o[t][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float mc[N], l[N];             // what stands for the maximum, in units of log2; this lane's part of the sum
#pragma unroll
  for (int n = 0; n < N; ++n) {
    mc[n] = -1e30f;
    l[n] = 0.f;
  }

  if (t1 > 0) {
    const unsigned lds = lds_address(smem);
    // ---- loads: tiles `lk` of K and `lv` of V next; after the last one it repeats
    int lk = 0, lv = 0;
    const char* kb = reinterpret_cast<const char*>(a.k + ((long)b * a.Skv * a.Hk + kvh) * DQK);
    const char* vb = reinterpret_cast<const char*>(a.v + ((long)b * a.Skv * a.Hk + kvh) * DV);
    unsigned koff[DQK / 32], voff[DV / 32];
    // (`here` in what is seldom run: nothing of it is kept in registers meanwhile)
    auto k_offsets = [&]() {       // rows beyond Skv: the last one
      const int have = min(a.Skv - lk * 64, 64);
      int lane = threadIdx.x & 63;
      here(lane);
#pragma unroll
      for (int i = 0; i < DQK / 32; ++i) {
        const int p = (4 * i + wid) * 64 + lane, row = p / (DQK / 8), slot = p % (DQK / 8);
        koff[i] = (unsigned)min(row, have - 1) * (unsigned)(a.Hk * T::KR) + ((slot ^ place(T::KR, row)) << 4);
      }
    };
    auto v_offsets = [&]() {
      const int have = min(a.Skv - lv * 64, 64);
      int lane = threadIdx.x & 63;
      here(lane);
#pragma unroll
      for (int i = 0; i < DV / 32; ++i) {
        const int p = (4 * i + wid) * 64 + lane, row = p / (DV / 8), slot = p % (DV / 8);
        voff[i] = (unsigned)min(row, have - 1) * (unsigned)(a.Hk * T::VR) + ((slot ^ place(T::VR, row)) << 4);
      }
    };
    auto k_advance = [&]() {
      if (lk + 1 < t1) {
        ++lk;
        kb += 64l * a.Hk * T::KR;
        if (lk * 64 + 64 > a.Skv) k_offsets();
      }
    };
    auto v_advance = [&]() {
      if (lv + 1 < t1) {
        ++lv;
        vb += 64l * a.Hk * T::VR;
        if (lv * 64 + 64 > a.Skv) v_offsets();
      }
    };
    const unsigned lw = lds + wid * 1024;
    unsigned to_k = lw, to_v = lw;               // the buffers that are loaded
    auto load_k = [&](auto i_) __attribute__((always_inline)) {
      constexpr int i = decltype(i_)::value;
      gt::load_lds(to_k, i * 4096, koff[i], kb);
    };
    auto load_v = [&](auto i_) __attribute__((always_inline)) {
      constexpr int i = decltype(i_)::value;
      gt::load_lds(to_v, KT + i * 4096, voff[i], vb);
    };
    k_offsets();
    v_offsets();
    unrolled<DQK / 32>(load_k);
    k_advance();
    to_k += BUF;
    unrolled<DV / 32>(load_v);
    v_advance();
    to_v += BUF;
    unrolled<DQK / 32>(load_k);
    k_advance();
    to_k += BUF;

    // ---- reads
    // windows: rows of K by 32 columns, columns of V by 16
    unsigned kr[DQK / 32], vc[DV / 16];
    const int crow = 4 * g + (i16 >> 2), piece = (i16 & 3) >> 1;
#pragma unroll
    for (int s = 0; s < DQK / 32; ++s) kr[s] = lds + i16 * T::KR + (((4 * s + g) ^ place(T::KR, i16)) << 4);
#pragma unroll
    for (int t = 0; t < DV / 16; ++t)
      vc[t] = lds + KT + crow * T::VR + (((2 * t + piece) ^ place(T::VR, crow)) << 4) + (i16 & 1) * 8;
    typedef __attribute__((address_space(3))) bf16x8_t* row_ptr;
    typedef __attribute__((address_space(3))) bf16x4_t* col_ptr;
    bf16x8_t ring[RING];
    // fragment f of a step into its place; HALF: of the tile that the windows are at; part 0 and 1:
    // halves of the summed index (columns)
    auto read = [&](auto f_, auto part_, auto half_) __attribute__((always_inline)) {
      constexpr int f = decltype(f_)::value, part = decltype(part_)::value, HALF = decltype(half_)::value;
      bf16x8_t& d = ring[f % RING];
      if constexpr (f < F1) {
        if constexpr (part == 0) d = *(row_ptr)(uintptr_t)(kr[f / 2] + HALF * 32 * T::KR + f % 2 * 16 * T::KR);
      } else {
        const bf16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (col_ptr)(uintptr_t)(vc[f - F1] + HALF * 32 * T::VR + part * 16 * T::VR));
#pragma unroll
        for (int j = 0; j < 4; ++j) d[4 * part + j] = v[j];
      }
    };

    f32x4_t s[2][2][N];                          // half, 16 keys, 16 rows
    u32x4_t e[2][N];                             // P as an operand
    float ls[N];                                 // the step's sums
    int by_key = BUF, by_col = 0, kbuf = 0, vbuf = 0;
    auto hide = [&](f32x4_t (&x)[2][N], int key0) __attribute__((always_inline)) {
      int first = qpos - 4 * g, g4 = 4 * g;
      here(first);
      here(g4);
#pragma unroll
      for (int z = 0; z < 8 * N; ++z) {
        const int zk = z / (4 * N), zq = z / 4 % N, zr = z % 4, key = key0 + zk * 16 + zr;
        if ((a.causal && key > first + 16 * zq) || key + g4 >= a.Skv) x[zk][zq][zr] = -INFINITY;
      }
    };

    auto maximum = [&](const f32x4_t (&x)[2][N], int n) __attribute__((always_inline)) {
      float m = x[0][n][0];
#pragma unroll
      for (int z = 1; z < 8; ++z) m = fmaxf(m, x[z / 4][n][z % 4]);
      m = fmaxf(m, __shfl_xor(m, 16));
      return fmaxf(m, __shfl_xor(m, 32));
    };

    // a step: SUB is the half that goes through the exponential; mask: the next one has keys that
    // some row must not see, from key0 on
    auto step = [&](auto sub_, bool mask, int key0) __attribute__((always_inline)) {
      constexpr int SUB = decltype(sub_)::value, O = 1 - SUB;
      using Sub = std::integral_constant<int, SUB>;
      using Oth = std::integral_constant<int, O>;
      using I0 = std::integral_constant<int, 0>;
      using I1 = std::integral_constant<int, 1>;
      __builtin_amdgcn_sched_barrier(0);
      unrolled<SLOTS>([&](auto m_) __attribute__((always_inline)) {
        constexpr int m = decltype(m_)::value, f = m / N, n = m % N;
        if constexpr (SUB == 0 && m == N * (F - RING + 1)) {
          wait_loads();            // the next tile's K, this one's V
          barrier();               // and the buffers of K and V before them are read
          __builtin_amdgcn_sched_barrier(0);
        }
        const bf16x8_t x = ring[f % RING];
        if constexpr (f < F1) {
          if constexpr (f < 2) mfma_first(s[O][f % 2][n], x, qf[n][0]);
          else mfma_next(s[O][f % 2][n], x, qf[n][f / 2]);
        } else {
          gt::mfma(o[f - F1][n], x, __builtin_bit_cast(bf16x8_t, e[O][n]));
        }
        // the fragment RING - 1 on, into the place of the last one
        constexpr int next = f + RING - 1;
        if constexpr (n == 0) {
          if constexpr (next < F) read(std::integral_constant<int, next>{}, I0{}, Oth{});
          else read(std::integral_constant<int, next - F>{}, I0{}, Sub{});
        } else if constexpr (n == 1 && next < F) {
          read(std::integral_constant<int, next>{}, I1{}, Oth{});
        }
        if constexpr (m == N * F1 + 4)
          if (mask) hide(s[O], key0);
        spread<m, SLOTS - 2, T::OPS>([&](auto i_) __attribute__((always_inline)) {
          constexpr int i = decltype(i_)::value, E = T::E;
          constexpr int v = i / 3 - i % 3, k = v / (4 * N), q = v / 4 % N, r = v % 4;
          if constexpr (i < T::EXPS) {
            if constexpr (v >= 0 && v < E) {
              if constexpr (i % 3 == 2) {
                if constexpr (k == 0 && r == 0) ls[q] = s[SUB][k][q][r];
                else ls[q] += s[SUB][k][q][r];
                here(ls[q]);
              } else {
                float y = s[SUB][k][q][r];
                if constexpr (i % 3 == 0) y = fmaf(y, c, -mc[q]);
                else y = __builtin_amdgcn_exp2f(y);
                here(y);
                s[SUB][k][q][r] = y;
              }
            }
          } else {
            constexpr int w = i - T::EXPS, wk = w / (2 * N), wq = w / 2 % N, wr = w % 2 * 2;   // pair w
            unsigned y = pair(s[SUB][wk][wq][wr], s[SUB][wk][wq][wr + 1]);
            here(y);
            e[SUB][wq][wk * 2 + wr / 2] = y;
          }
        });
        if constexpr (SUB == 0) {
          // on to the next tile's rows of K, once this one's are read; and to this tile's columns
          constexpr int A = N * (F1 - RING) + 4, B = N * (F - RING) + 4;
          if constexpr (m >= A && m - A < DQK / 32) kr[m - A] += by_key;
          if constexpr (m >= B && m - B < DV / 16) vc[m - B] += by_col;
          constexpr int L = N * (F - RING + 1) + 1, EVERY = (SLOTS - L) / (DQK / 32);
          if constexpr (m >= L && (m - L) % EVERY == 0 && (m - L) / EVERY < DQK / 32)
            load_k(std::integral_constant<int, (m - L) / EVERY>{});
        } else {
          constexpr int EVERY = SLOTS / 2 / (DV / 32);
          if constexpr (m % EVERY == 2 && m / EVERY < DV / 32) load_v(std::integral_constant<int, m / EVERY>{});
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    // the end of a step: `mask` and key0 are those of its own keys
    auto finish = [&](auto sub_, bool mask, int key0) __attribute__((always_inline)) {
      constexpr int SUB = decltype(sub_)::value;
      float most = 0.f;
#pragma unroll
      for (int n = 0; n < N; ++n) {
        ls[n] += l[n];
        most = n == 0 ? ls[n] : fmaxf(most, ls[n]);
      }
      if (__any(most > 0x1p32f)) {
        f32x4_t (&x)[2][N] = s[SUB];
#pragma unroll
        for (int f = 0; f < F1; ++f) {           // (the windows are a tile on)
          const bf16x8_t y = *(row_ptr)(uintptr_t)(kr[f / 2] - by_key + SUB * 32 * T::KR + f % 2 * 16 * T::KR);
#pragma unroll
          for (int n = 0; n < N; ++n) {
            if (f < 2) mfma_first(x[f % 2][n], y, qf[n][0]);
            else mfma_next(x[f % 2][n], y, qf[n][f / 2]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        gt::settle();
        if (mask) hide(x, key0);
#pragma unroll
        for (int n = 0; n < N; ++n) {
          float all = fmaxf(l[n], 1.f);          // (a sum of many, too, starts anew at 1)
          all = fmaxf(all, __shfl_xor(all, 16));
          all = fmaxf(all, __shfl_xor(all, 32));
          const float now = fmaxf(mc[n] + __builtin_amdgcn_logf(all), maximum(x, n) * c);
          const float alpha = __builtin_amdgcn_exp2f(mc[n] - now);
          float sum = l[n] * alpha;
#pragma unroll
          for (int z = 0; z < 8; ++z) {
            const float y = __builtin_amdgcn_exp2f(fmaf(x[z / 4][n][z % 4], c, -now));
            sum += y;
            x[z / 4][n][z % 4] = y;
          }
          mc[n] = now;
          ls[n] = sum;
#pragma unroll
          for (int w = 0; w < 4; ++w)
            e[SUB][n][w] = pair(x[w / 2][n][w % 2 * 2], x[w / 2][n][w % 2 * 2 + 1]);
#pragma unroll
          for (int t = 0; t < DV / 16; ++t) {
            f32x4_t y = o[t][n];
            here(y);
            y *= alpha;
            here(y);
            o[t][n] = y;
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        gt::settle();
      }
#pragma unroll
      for (int n = 0; n < N; ++n) l[n] = ls[n];
    };
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;

    wait_loads();
    barrier();
    // S of the first half with its maximum, and the operands of the first step
    unrolled<F1>([&](auto f_) __attribute__((always_inline)) {
      constexpr int f = decltype(f_)::value;
      read(f_, P0{}, P0{});
#pragma unroll
      for (int n = 0; n < N; ++n) {
        if constexpr (f < 2) mfma_first(s[0][f][n], ring[f % RING], qf[n][0]);
        else mfma_next(s[0][f % 2][n], ring[f % RING], qf[n][f / 2]);
      }
    });
    gt::settle();
    if (masked(0)) hide(s[0], 0);
#pragma unroll
    for (int n = 0; n < N; ++n) {
      mc[n] = fmaxf(mc[n], maximum(s[0], n) * c);
      e[1][n] = u32x4_t{0, 0, 0, 0};
    }
    unrolled<RING - 1>([&](auto f_) __attribute__((always_inline)) { read(f_, P0{}, P1{}); });
    gt::settle();

#pragma unroll 1
    for (int t = 0; t < t1; ++t) {
      step(P0{}, masked(t), t * 64 + 32);
      finish(P0{}, masked(t), t * 64);
      step(P1{}, masked(t + 1), t * 64 + 64);
      finish(P1{}, masked(t), t * 64 + 32);
      kbuf = kbuf == 2 ? 0 : kbuf + 1;
      by_key = kbuf == 2 ? -2 * BUF : BUF;
      if (t > 0) vbuf = vbuf == 2 ? 0 : vbuf + 1;
      by_col = vbuf == 2 ? -2 * BUF : BUF;
      to_k = to_k == lw + 2 * BUF ? lw : to_k + BUF;
      to_v = to_v == lw + 2 * BUF ? lw : to_v + BUF;
      k_advance();
      v_advance();
    }
    // the last half's values
    unrolled<F>([&](auto f_) __attribute__((always_inline)) {
      constexpr int f = decltype(f_)::value;
      if constexpr (f >= F1) {
        read(f_, P0{}, P1{});
        read(f_, P1{}, P1{});
#pragma unroll
        for (int n = 0; n < N; ++n) gt::mfma(o[f - F1][n], ring[f % RING], __builtin_bit_cast(bf16x8_t, e[1][n]));
      }
    });
    wait_loads();
    gt::settle();
    barrier();
  }

  // ---- normalise, then to memory in whole rows, through the wave's part of LDS. A sink is one more logit
  // in the denominator, without a key.
  constexpr int CH = DV / 8;
  char* mine = smem + wid * T::ROWS * T::VR;
  bf16* dst = a.out + (((long)b * a.Sq + q0) * a.Hq + h) * DV;
#pragma unroll
  for (int n = 0; n < N; ++n) {
    float ls = l[n] + __shfl_xor(l[n], 16);
    ls += __shfl_xor(ls, 32);
    if (a.sink) ls += __builtin_amdgcn_exp2f(bf2f(a.sink[h]) * LOG2E - mc[n]);
    const float inv = ls > 0.f ? 1.f / ls : 0.f;
    const int row = n * 16 + i16;
    if (g == 0 && q0 + row < a.Sq)
      a.lse[((long)b * a.Hq + h) * a.Sq + q0 + row] = ls > 0.f ? mc[n] * LN2 + __logf(ls) : -1e30f;
#pragma unroll
    for (int t = 0; t < DV / 16; ++t) {
      bf16x4_t w;
#pragma unroll
      for (int r = 0; r < 4; ++r) w[r] = (__bf16)(o[t][n][r] * inv);
      const int ch = (2 * t + (g >> 1)) ^ place(T::VR, row);
      *reinterpret_cast<bf16x4_t*>(mine + row * T::VR + (ch << 4) + (g & 1) * 8) = w;
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    // a wave reads what it wrote itself
  for (int p = lane; p < T::ROWS * CH; p += 64) {
    const int row = p / CH, ch = p % CH;
    if (q0 + row < a.Sq)
      *reinterpret_cast<uint4*>(dst + (long)row * a.Hq * DV + ch * 8) =
          *reinterpret_cast<const uint4*>(mine + row * T::VR + ((ch ^ place(T::VR, row)) << 4));
  }
}

}  // namespace fa
}  // namespace amd_ops
