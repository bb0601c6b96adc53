// dQ of the flash-attention backward for values of 128 columns, keys of 128 or 192 (gfx950); included
// by flash_attn_bwd.hip.
//
// A wave has 16 N rows of Q and dO with their gradients (N = 4, or 3 with keys of 192: what the AGPRs hold),
// so that an operand from LDS serves N products; tiles of 64 rows of K and V pass by. Instructions
// are in a given order, as in flash_dkv.h. Over half tiles h of 32 keys a step has
//   dP(h) = V dO^T - delta, S(h + 1) = K Q^T, dQ^T += K^T dS(h - 1)
// and behind the MFMAs first the exponentials of h, whose scores are there, then, with dP(h)
// complete, dS(h). S[k][q] leaves a lane (q = lane & 15, g = lane >> 4) with keys 4 g + 0..3 of 16: two such
// tiles are the 8 summed indices of an operand of dQ^T, as they lie.
//
// Three buffers of a tile: the one whose columns of K are last read, the one at hand, whose rows of V
// are read first, and the next. One barrier a tile.
//
// Two waves a SIMD of 32 rows each, in the compiler's order, read twice as much LDS for a product
// (66% of the time in the matrix cores, LDS as busy). 1 x 16384, 32/8 heads of 128: 2.76 -> 2.3 ms;
// 2 x 3001, 16 heads (192, 128): 222 -> 140 us (there the 32 rows were one wave a SIMD).
#pragma once

#include "flash_ordered.h"

namespace amd_ops {
namespace fa {

template <int DQK, int DV>
struct DqTile {
  static constexpr int N = DQK == 128 ? 4 : 3, ROWS = 16 * N, BM = 4 * ROWS;   // rows of a wave, a workgroup
  static constexpr int KR = DQK * 2, VR = DV * 2;                        // bytes of a row
  static constexpr int KT = 64 * KR, VT = 64 * VR, BUF = KT + VT, SMEM = 3 * BUF;
  // fragments of a step: rows of V, rows of K, columns of K
  static constexpr int F1 = DV / 16, F2 = F1 + DQK / 16, F = F2 + DQK / 16;
  // rows of dO that the AGPRs have room for beside the gradients and Q, 32 columns of 16 each
  static constexpr int DO_AGPRS = (256 - DQK / 16 * N * 4 - DQK / 32 * N * 4) / 4;
  static_assert(F % 8 == 0 && SMEM <= 160 * 1024 && BM * KR <= SMEM, "8 places, three tiles; the result in them");
};

template <int DQK, int DV, class Args>
__global__ __launch_bounds__(256, 1) void bwd_dq_ordered_kernel(const Args a) {
  using T = DqTile<DQK, DV>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int BUF = T::BUF, KT = T::KT, F = T::F, N = T::N, SLOTS = F * N;
  const Place at = place_block((a.Sq + T::BM - 1) / T::BM, a.Hq, a.B, a.causal);
  const int lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = at.head, b = at.batch, kvh = h / (a.Hq / a.Hk);
  const int qblk = at.tile * T::BM, q0 = qblk + wid * T::ROWS;
  const float c = a.scale * LOG2E;

  // ---- the wave's rows of Q and dO, columns of S, and what goes with them
  bf16x8_t qf[N][DQK / 32], of[N][DV / 32];
  float l2[N];
  f32x4_t nd[N];
#pragma unroll
  for (int t = 0; t < N; ++t) {
    const int row = min(q0 + 16 * t + i16, a.Sq - 1);        // rows beyond Sq are not stored
    const long at_row = ((long)b * a.Sq + row) * a.Hq + h;
#pragma unroll
    for (int s = 0; s < DQK / 32; ++s)
      qf[t][s] = *reinterpret_cast<const bf16x8_t*>(a.q + at_row * DQK + s * 32 + g * 8);
#pragma unroll
    for (int s = 0; s < DV / 32; ++s)
      of[t][s] = *reinterpret_cast<const bf16x8_t*>(a.dout + at_row * DV + s * 32 + g * 8);
    const float* st = a.stats + ((long)b * a.Hq + h) * a.sp + row;
    l2[t] = st[0];
    const float d = st[a.plane];
    nd[t] = f32x4_t{d, d, d, d};
  }
  const int qpos = a.q_start + q0 + i16;

  // ---- key tiles that some row of the block sees
  const int last = a.q_start + min(qblk + T::BM, a.Sq) - 1, all = (a.Skv + 63) / 64;
  const int t1 = a.causal ? min(last / 64 + 1, all) : all;
  const int t_diag = a.causal ? (a.q_start + q0 + 1) / 64 : all;

  f32x4_t dq[DQK / 16][N];
#pragma unroll
  for (int t = 0; t < DQK / 16; ++t)
#pragma unroll
    for (int n = 0; n < N; ++n) dq[t][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  if (t1 > 0) {
    const unsigned lds = lds_address(smem);
    // ---- loads: tile `lt` next; after the last one it repeats
    int lt = 0;
    const char* kb = reinterpret_cast<const char*>(a.k + ((long)b * a.Skv * a.Hk + kvh) * DQK);
    const char* vb = reinterpret_cast<const char*>(a.v + ((long)b * a.Skv * a.Hk + kvh) * DV);
    unsigned koff[DQK / 32], voff[DV / 32];
    auto offsets = [&]() {       // rows beyond Skv: the last one
      const int have = min(a.Skv - lt * 64, 64);
#pragma unroll
      for (int i = 0; i < DQK / 32; ++i) {
        const int p = (4 * i + wid) * 64 + lane, row = p / (DQK / 8), slot = p % (DQK / 8);
        koff[i] = (unsigned)min(row, have - 1) * (unsigned)(a.Hk * T::KR) + ((slot ^ place(T::KR, row)) << 4);
      }
#pragma unroll
      for (int i = 0; i < DV / 32; ++i) {
        const int p = (4 * i + wid) * 64 + lane, row = p / (DV / 8), slot = p % (DV / 8);
        voff[i] = (unsigned)min(row, have - 1) * (unsigned)(a.Hk * T::VR) + ((slot ^ place(T::VR, row)) << 4);
      }
    };
    auto advance = [&]() {
      if (lt + 1 < t1) {
        ++lt;
        kb += 64l * a.Hk * T::KR;
        vb += 64l * a.Hk * T::VR;
        if (lt * 64 + 64 > a.Skv) offsets();
      }
    };
    const unsigned lw = lds + wid * 1024;
    unsigned to = lw;                            // the buffer that is loaded
    constexpr int LOADS = (DQK + DV) / 32;
    auto load = [&](auto i_) __attribute__((always_inline)) {
      constexpr int i = decltype(i_)::value;
      if constexpr (i < DQK / 32) gt::load_lds(to, i * 4096, koff[i], kb);
      else gt::load_lds(to, KT + (i - DQK / 32) * 4096, voff[i - DQK / 32], vb);
    };
    offsets();
#pragma unroll 1
    for (int u = 0; u < 2; ++u) {
      unrolled<LOADS>(load);
      to += BUF;
      advance();
    }

    // ---- reads
    // windows: rows of V and K by 32 columns, columns of K by 16
    unsigned vr[DV / 32], kr[DQK / 32], kc[DQK / 16];
    const int crow = 4 * g + (i16 >> 2), piece = (i16 & 3) >> 1;
#pragma unroll
    for (int s = 0; s < DV / 32; ++s) vr[s] = lds + KT + i16 * T::VR + (((4 * s + g) ^ place(T::VR, i16)) << 4);
#pragma unroll
    for (int s = 0; s < DQK / 32; ++s) kr[s] = lds + i16 * T::KR + (((4 * s + g) ^ place(T::KR, i16)) << 4);
#pragma unroll
    for (int t = 0; t < DQK / 16; ++t)
      kc[t] = lds + crow * T::KR + (((2 * t + piece) ^ place(T::KR, crow)) << 4) + (i16 & 1) * 8;
    typedef __attribute__((address_space(3))) bf16x8_t* row_ptr;
    typedef __attribute__((address_space(3))) bf16x4_t* col_ptr;
    bf16x8_t ring[8];
    // fragment f of a step into its place. Rows: by 32 columns, then 16 rows. VS, KS, CS: half of the
    // tile that the windows are at; part 0 and 1: halves of the summed index (columns)
    auto read = [&](auto f_, auto part_, auto vs_, auto ks_, auto cs_) __attribute__((always_inline)) {
      constexpr int f = decltype(f_)::value, part = decltype(part_)::value;
      constexpr int VS = decltype(vs_)::value, KS = decltype(ks_)::value, CS = decltype(cs_)::value;
      bf16x8_t& d = ring[f % 8];
      if constexpr (f < T::F2) {
        if constexpr (part == 0) {
          constexpr int n = f < T::F1 ? f : f - T::F1, R = f < T::F1 ? T::VR : T::KR, S = f < T::F1 ? VS : KS;
          const unsigned p = f < T::F1 ? vr[n / 2 % (DV / 32)] : kr[n / 2 % (DQK / 32)];
          d = *(row_ptr)(uintptr_t)(p + S * 32 * R + n % 2 * 16 * R);
        }
      } else {
        const bf16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (col_ptr)(uintptr_t)(kc[f - T::F2] + CS * 32 * T::KR + part * 16 * T::KR));
#pragma unroll
        for (int j = 0; j < 4; ++j) d[4 * part + j] = v[j];
      }
    };

    f32x4_t s[2][2][N], dp[2][N];                // half, 16 keys, 16 rows
    u32x4_t e[2][N];                             // dS as an operand
    int by_key = BUF, by_col = 0, kbuf = 0, cbuf = 0;

    // a step: SUB is the half whose dS is formed
    auto step = [&](auto sub_, int t, bool mask) __attribute__((always_inline)) {
      constexpr int SUB = decltype(sub_)::value, O = 1 - SUB;
      using Sub = std::integral_constant<int, SUB>;
      using Oth = std::integral_constant<int, O>;
      using I0 = std::integral_constant<int, 0>;
      using I1 = std::integral_constant<int, 1>;
      if constexpr (SUB == 1) {
        wait_loads();              // the next tile; and the columns of the tile before are read
        asm volatile("s_waitcnt lgkmcnt(7)\n\ts_barrier" ::: "memory");
      }
      __builtin_amdgcn_sched_barrier(0);
      unrolled<SLOTS>([&](auto m_) __attribute__((always_inline)) {
        constexpr int m = decltype(m_)::value, f = m / N, n = m % N;
        const bf16x8_t x = ring[f % 8];
        if constexpr (f < T::F1) {
          if constexpr (n * (DV / 32) + f / 2 < T::DO_AGPRS) {
            if constexpr (f < 2) mfma_first(dp[f % 2][n], x, of[n][0], nd[n]);
            else mfma_next(dp[f % 2][n], x, of[n][f / 2]);
          } else {
            if constexpr (f < 2) mfma_first_v(dp[f % 2][n], x, of[n][0], nd[n]);
            else mfma_next_v(dp[f % 2][n], x, of[n][f / 2]);
          }
        } else if constexpr (f < T::F2) {
          constexpr int k = f - T::F1;
          if constexpr (k < 2) mfma_first(s[O][k % 2][n], x, qf[n][0]);
          else mfma_next(s[O][k % 2][n], x, qf[n][k / 2]);
        } else {
          gt::mfma(dq[f - T::F2][n], x, __builtin_bit_cast(bf16x8_t, e[O][n]));
        }
        // the fragment 7 on, into the place of the last one
        if constexpr (n == 0) {
          if constexpr (f + 7 < F) read(std::integral_constant<int, f + 7>{}, I0{}, Sub{}, Oth{}, Oth{});
          else read(std::integral_constant<int, f + 7 - F>{}, I0{}, Oth{}, I0{}, I0{});
        } else if constexpr (n == 1 && f + 7 < F) {
          read(std::integral_constant<int, f + 7>{}, I1{}, Sub{}, Oth{}, Oth{});
        }
        // 28 N operations: multiplications and additions with their exponentials, then products
        // with the roundings
        constexpr int E = 8 * N, OPS = E * 7 / 2;
        spread<m, SLOTS, OPS>([&](auto i_) __attribute__((always_inline)) {
          constexpr int i = decltype(i_)::value;
          if constexpr (i < 2 * E) {
            constexpr int v = i / 2, k = v / (4 * N), q = v / 4 % N, r = v % 4;
            float y = s[SUB][k][q][r];
            if constexpr (i % 2 == 0) y = fmaf(y, c, -l2[q]);
            else y = __builtin_amdgcn_exp2f(y);
            here(y);
            s[SUB][k][q][r] = y;
            if (i == 2 * E - 1 && mask) {
#pragma unroll
              for (int z = 0; z < E; ++z) {
                const int zk = z / (4 * N), zq = z / 4 % N, zr = z % 4;
                const int key = t * 64 + SUB * 32 + zk * 16 + 4 * g + zr;
                if ((a.causal && key > qpos + 16 * zq) || key >= a.Skv)
                  s[SUB][zk][zq][zr] = 0.f;
              }
            }
          } else {
            constexpr int j = i - 2 * E, w = j / 3, k = w / (2 * N), q = w / 2 % N, r = w % 2 * 2;   // pair w
            if constexpr (j % 3 < 2) {
              float y = dp[k][q][r + j % 3] * s[SUB][k][q][r + j % 3];
              here(y);
              dp[k][q][r + j % 3] = y;
            } else {
              typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
              unsigned y = __builtin_bit_cast(unsigned, bf16x2_t{(__bf16)dp[k][q][r], (__bf16)dp[k][q][r + 1]});
              here(y);
              e[SUB][q][k * 2 + r / 2] = y;
            }
          }
        });
        if constexpr (SUB == 0) {
          // on to the next tile's rows of K, once this one's are read; and to this tile's columns
          constexpr int A = N * (T::F2 - 7) + 4, B = N * (F - 7) + 4;
          if constexpr (m >= A && m - A < DQK / 32) kr[m - A] += by_key;
          if constexpr (m >= B && m - B < DQK / 16) kc[m - B] += by_col;
        } else {
          // on to the next tile's rows of V
          constexpr int A = N * (T::F1 - 7) + 4, EVERY = SLOTS / LOADS;
          if constexpr (m >= A && m - A < DV / 32) vr[m - A] += by_key;
          if constexpr (m % EVERY == 2 && m / EVERY < LOADS) load(std::integral_constant<int, m / EVERY>{});
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;

    wait_loads();
    barrier();
    // S of the first half and the operands of the first step
    unrolled<DQK / 16>([&](auto f_) __attribute__((always_inline)) {
      constexpr int k = decltype(f_)::value;
      using Frag = std::integral_constant<int, T::F1 + k>;
      read(Frag{}, P0{}, P0{}, P0{}, P0{});
#pragma unroll
      for (int n = 0; n < N; ++n) {
        if constexpr (k < 2) mfma_first(s[0][k][n], ring[Frag::value % 8], qf[n][0]);
        else mfma_next(s[0][k % 2][n], ring[Frag::value % 8], qf[n][k / 2]);
      }
    });
#pragma unroll
    for (int n = 0; n < N; ++n) e[1][n] = u32x4_t{0, 0, 0, 0};
    unrolled<7>([&](auto f_) __attribute__((always_inline)) { read(f_, P0{}, P0{}, P0{}, P0{}); });
    gt::settle();

#pragma unroll 1
    for (int t = 0; t < t1; ++t) {
      const bool mask = t >= t_diag || t * 64 + 64 > a.Skv;
      step(P0{}, t, mask);
      by_col = t == 0 ? BUF : by_col;
      step(P1{}, t, mask);
      kbuf = kbuf == 2 ? 0 : kbuf + 1;
      by_key = kbuf == 2 ? -2 * BUF : BUF;
      if (t > 0) cbuf = cbuf == 2 ? 0 : cbuf + 1;
      by_col = cbuf == 2 ? -2 * BUF : BUF;
      to = to == lw + 2 * BUF ? lw : to + BUF;
      advance();
    }
    // the last half's gradients
    unrolled<F>([&](auto f_) __attribute__((always_inline)) {
      constexpr int f = decltype(f_)::value;
      if constexpr (f >= T::F2) {
        read(f_, P0{}, P0{}, P0{}, P1{});
        read(f_, P1{}, P0{}, P0{}, P1{});
#pragma unroll
        for (int n = 0; n < N; ++n) gt::mfma(dq[f - T::F2][n], ring[f % 8], __builtin_bit_cast(bf16x8_t, e[1][n]));
      }
    });
    wait_loads();
    gt::settle();
    barrier();
  }

  // ---- to memory in whole rows, through the wave's part of LDS
  constexpr int CH = DQK / 8;
  char* mine = smem + wid * T::ROWS * T::KR;
  bf16* dst = a.dq + (((long)b * a.Sq + q0) * a.Hq + h) * DQK;
#pragma unroll
  for (int n = 0; n < N; ++n)
#pragma unroll
    for (int t = 0; t < DQK / 16; ++t) {
      bf16x4_t w;
#pragma unroll
      for (int r = 0; r < 4; ++r) w[r] = (__bf16)(dq[t][n][r] * a.scale);
      const int row = n * 16 + i16, ch = (2 * t + (g >> 1)) ^ place(T::KR, row);
      *reinterpret_cast<bf16x4_t*>(mine + row * T::KR + (ch << 4) + (g & 1) * 8) = w;
    }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    // a wave reads what it wrote itself
  for (int p = lane; p < T::ROWS * CH; p += 64) {
    const int row = p / CH, ch = p % CH;
    if (q0 + row < a.Sq)
      *reinterpret_cast<uint4*>(dst + (long)row * a.Hq * DQK + ch * 8) =
          *reinterpret_cast<const uint4*>(mine + row * T::KR + ((ch ^ place(T::KR, row)) << 4));
  }
}

}  // namespace fa
}  // namespace amd_ops
