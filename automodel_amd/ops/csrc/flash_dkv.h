// dK and dV of the flash-attention backward for values of 128 columns, keys of 128 or 192 (gfx950);
// included by flash_attn_bwd.hip.
//
// A workgroup has 128 rows of K and V, a wave 32 of them with their gradients (accumulators and
// the rows themselves in AGPRs), so that one wave has a SIMD to itself; tiles of 64 rows of Q and dO
// pass by. The wave's instructions issue in order, and what the compiler makes of the loop
// leaves the matrix cores idle while it waits for LDS and forms exponentials (39% busy). So the
// order is given here. Over half tiles h of 32 rows a step has
//   S(h + 1) = Q K^T, dP(h + 1) = dO V^T - delta     32 MFMAs of 16 cycles (40 with keys of 192)
//   dV += dO^T P(h - 1), dK += Q^T dS(h - 1)         32 (40)
// and behind each MFMA one vector instruction of P(h) and dS(h) and at most one LDS read. An
// operand is read 13 MFMAs before its first use, into one of 8 places (LDS has room for 15
// requests of a wave).
//
// S[q][k] leaves a lane (k = lane & 15, g = lane >> 4) with rows 4 g + 0..3 of 16; two such tiles are
// the 8 summed indices of an operand of the next products, whose other operand is read in
// the same order, rows 4 g + 0..3 and 16 + 4 g + 0..3 (transposing LDS reads).
//
// Four buffers of a tile: the one whose columns are last read, the one at hand, the next, whose
// rows are read first, and one that is loaded, with one barrier a tile. Keys of 192 have three:
// the barrier waits for the last columns, just before the next rows are read.
//
// Now 59% of the time in the matrix cores (1742 cycles for a step of 1024), LDS about as busy: a
// step's 52 reads of 4 waves take 950 cycles, its share of the loads 130 and more. 1 x
// 16384, 32/8 heads of 128: 5.45 -> 3.75 ms (3.96 with each workgroup at its own place in Q and dO,
// and conflicts in the reads of rows); 2 x 3001, 16 heads (192, 128): 283 -> 203 us.
#pragma once

#include "flash_ordered.h"

namespace amd_ops {
namespace fa {

template <int DQK, int DV>
struct DkvTile {
  static constexpr int QR = DQK * 2, OR = DV * 2;                        // bytes of a row
  static constexpr int QT = 64 * QR, OT = 64 * OR, BUF = QT + OT + 1024;   // Q, dO, statistics
  static constexpr int BUFS = 4 * BUF <= 160 * 1024 ? 4 : 3, SMEM = BUFS * BUF;
  // fragments of a step: rows of Q and dO, columns of dO and Q
  static constexpr int F1 = DQK / 16, F2 = F1 + DV / 16, F3 = F2 + DV / 16, F = F3 + DQK / 16;
  static_assert(DQK % 64 == 0 && DV % 64 == 0 && SMEM <= 160 * 1024, "whole tiles, 8 places for operands");
};

template <int DQK, int DV, bool VARLEN, class Args>
__global__ __launch_bounds__(256, 1) void bwd_dkv_ordered_kernel(const Args a) {
  using T = DkvTile<DQK, DV>;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  constexpr int BUF = T::BUF, BUFS = T::BUFS, QT = T::QT, F = T::F;
  const Place at = place_block((a.Skv + 127) / 128, a.Hk, a.B, false);
  const int lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kvh = at.head, b = at.batch, G = a.Hq / a.Hk;
  const int kvb = at.tile * 128, kv0 = kvb + wid * 32;
  const float c = a.scale * LOG2E;

  // ---- the wave's rows of K and V: columns of S
  bf16x8_t kf[2][DQK / 32], vf[2][DV / 32];
  int kend[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int row = min(kv0 + 16 * t + i16, a.Skv - 1);      // rows beyond Skv are not stored
    const long at_row = ((long)b * a.Skv + row) * a.Hk + kvh;
#pragma unroll
    for (int s = 0; s < DQK / 32; ++s)
      kf[t][s] = *reinterpret_cast<const bf16x8_t*>(a.k + at_row * DQK + s * 32 + g * 8);
#pragma unroll
    for (int s = 0; s < DV / 32; ++s)
      vf[t][s] = *reinterpret_cast<const bf16x8_t*>(a.v + at_row * DV + s * 32 + g * 8);
    kend[t] = VARLEN ? a.doc_end[row] : 0;
  }

  // ---- query tiles that see some row of the block, for every head of the group
  const int j0 = a.causal && kvb > a.q_start ? (kvb - a.q_start) / 64 : 0;
  int j1 = (a.Sq + 63) / 64, end_w = 0x7fffffff;
  if (VARLEN) {
    const int de = __builtin_amdgcn_readfirstlane(a.doc_end[min(kvb + 128, a.Skv) - 1]);
    j1 = min(j1, (de - a.q_start + 63) / 64);
    end_w = __builtin_amdgcn_readfirstlane(a.doc_end[min(kv0, a.Skv - 1)]);
  }
  const int nt = max(j1 - j0, 0), total = nt * G;      // (j1 > j0 from here on)

  f32x4_t dk[DQK / 16][2], dv[DV / 16][2];
#pragma unroll
  for (int t = 0; t < DQK / 16; ++t) dk[t][0] = dk[t][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < DV / 16; ++t) dv[t][0] = dv[t][1] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  if (total > 0) {
    const unsigned lds = lds_address(smem);
    // ---- loads: tile j0 + lt of head `lh` of the group next; after the last one it repeats. All heads
    // of a tile, then the tile before: the workgroups of an XCD, whatever their first tile,
    // read the same ones at a time (5 GB of 17 missed L2 the other way round, now 1).
    int lt = nt - 1, lh = 0, left = total - 1;
    const long first = ((long)b * a.Sq + (j1 - 1) * 64) * a.Hq + kvh * G;
    const char* qb = reinterpret_cast<const char*>(a.q + first * DQK);
    const char* ob = reinterpret_cast<const char*>(a.dout + first * DV);
    const char* sb = reinterpret_cast<const char*>(
        a.stats + ((long)b * a.Hq + kvh * G) * a.sp + (j1 - 1) * 64 + (i16 * 4 + ((lane >> 4) & 1) * a.plane));
    const long back = 64l * a.Hq + G - 1, stat_back = 256 + (G - 1) * 4l * a.sp;
    unsigned qoff[DQK / 32], ooff[DV / 32];
    auto offsets = [&]() {       // rows beyond Sq: the last one
      const int have = min(a.Sq - (j0 + lt) * 64, 64);
#pragma unroll
      for (int h = 0; h < DQK / 32; ++h) {
        const int c = (4 * h + wid) * 64 + lane, row = c / (DQK / 8), slot = c % (DQK / 8);
        qoff[h] = (unsigned)min(row, have - 1) * (unsigned)(a.Hq * T::QR) + ((slot ^ place(T::QR, row)) << 4);
      }
#pragma unroll
      for (int h = 0; h < DV / 32; ++h) {
        const int c = (4 * h + wid) * 64 + lane, row = c / (DV / 8), slot = c % (DV / 8);
        ooff[h] = (unsigned)min(row, have - 1) * (unsigned)(a.Hq * T::OR) + ((slot ^ place(T::OR, row)) << 4);
      }
    };
    auto advance = [&]() {
      if (left > 0) {
        --left;
        if (++lh == G) {
          lh = 0;
          qb -= back * T::QR;
          ob -= back * T::OR;
          sb -= stat_back;
          if (--lt == nt - 2) offsets();         // only the last tile may be short
        } else {
          qb += T::QR;
          ob += T::OR;
          sb += 4l * a.sp;
        }
      }
    };
    const unsigned lw = lds + wid * 1024;
    unsigned to = lw;                            // the buffer that is loaded
    constexpr int LOADS = (DQK + DV) / 32;
    auto load = [&](auto i_) __attribute__((always_inline)) {
      constexpr int i = decltype(i_)::value;
      if constexpr (i < DQK / 32) gt::load_lds(to, i * 4096, qoff[i], qb);
      else gt::load_lds(to, QT + (i - DQK / 32) * 4096, ooff[i - DQK / 32], ob);
    };
    auto load_stats = [&]() {                    // 64 rows of both, lanes 32.. repeat
      if (wid == 0) load_lds16(to + QT + T::OT, sb);
    };
    offsets();
#pragma unroll 1
    for (int u = 0; u < BUFS - 1; ++u) {
      unrolled<LOADS>(load);
      load_stats();
      to += BUF;
      advance();
    }

    // ---- reads
    // windows: rows of Q and dO by 32 columns, columns of dO and Q by 16
    unsigned qr[DQK / 32], orow[DV / 32], oc[DV / 16], qc[DQK / 16];
    const int crow = 4 * g + (i16 >> 2), piece = (i16 & 3) >> 1;
#pragma unroll
    for (int s = 0; s < DQK / 32; ++s) qr[s] = lds + i16 * T::QR + (((4 * s + g) ^ place(T::QR, i16)) << 4);
#pragma unroll
    for (int s = 0; s < DV / 32; ++s)
      orow[s] = lds + QT + i16 * T::OR + (((4 * s + g) ^ place(T::OR, i16)) << 4);
#pragma unroll
    for (int t = 0; t < DV / 16; ++t)
      oc[t] = lds + QT + crow * T::OR + (((2 * t + piece) ^ place(T::OR, crow)) << 4) + (i16 & 1) * 8;
#pragma unroll
    for (int t = 0; t < DQK / 16; ++t)
      qc[t] = lds + crow * T::QR + (((2 * t + piece) ^ place(T::QR, crow)) << 4) + (i16 & 1) * 8;
    unsigned sw = lds + QT + T::OT + 16 * g;     // statistics of the tile at hand
    unsigned nw = sw;                            // and of the tile whose rows are read
    typedef __attribute__((address_space(3))) f32x4_t* stat_ptr;
    typedef __attribute__((address_space(3))) bf16x8_t* row_ptr;
    typedef __attribute__((address_space(3))) bf16x4_t* col_ptr;
    bf16x8_t ring[8];
    // fragment f of a step into its place. Rows: by 32 columns, then 16 rows. ROWS, COLS: half of
    // the tile that the windows are at; part 0 and 1: halves of the summed index (columns)
    auto read = [&](auto f_, auto part_, auto rows_, auto cols_) __attribute__((always_inline)) {
      constexpr int f = decltype(f_)::value, part = decltype(part_)::value;
      constexpr int ROWS = decltype(rows_)::value, COLS = decltype(cols_)::value;
      bf16x8_t& d = ring[f % 8];
      if constexpr (f < T::F2) {
        if constexpr (part == 0) {
          constexpr int n = f < T::F1 ? f : f - T::F1, R = f < T::F1 ? T::QR : T::OR;
          const unsigned at = f < T::F1 ? qr[n / 2 % (DQK / 32)] : orow[n / 2 % (DV / 32)];
          d = *(row_ptr)(uintptr_t)(at + ROWS * 32 * R + n % 2 * 16 * R);
        }
      } else {
        constexpr int n = f < T::F3 ? f - T::F2 : f - T::F3, R = f < T::F3 ? T::OR : T::QR;
        const unsigned at = f < T::F3 ? oc[n % (DV / 16)] : qc[n % (DQK / 16)];
        const bf16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (col_ptr)(uintptr_t)(at + COLS * 32 * R + part * 16 * R));
#pragma unroll
        for (int j = 0; j < 4; ++j) d[4 * part + j] = v[j];
      }
    };

    f32x4_t s[2][2][2], dp[2][2][2];             // half, 16 rows, 16 columns
    u32x4_t p[2][2], e[2][2];                    // P and dS as operands: half, 16 columns
    f32x4_t l2[2], nd[2];
    int ch = 0, qpos = a.q_start + (j1 - 1) * 64;      // head and first row of the tile at hand
    int by_row = BUF, by_col = 0, rbuf = 0, cbuf = 0;

    // a step: SUB is the half whose P and dS are formed
    auto step = [&](auto sub_, bool mask) __attribute__((always_inline)) {
      constexpr int SUB = decltype(sub_)::value, O = 1 - SUB;
      using Sub = std::integral_constant<int, SUB>;
      using Oth = std::integral_constant<int, O>;
      using I0 = std::integral_constant<int, 0>;
      using I1 = std::integral_constant<int, 1>;
      // rows of the other half: of this tile (SUB 0) or the next one; columns of the other half:
      // of the tile before, or of this one
      if constexpr (SUB == 1 && BUFS == 4) {
        wait_loads();              // the tile after next; and the columns of the tile before are read
        asm volatile("s_waitcnt lgkmcnt(7)\n\ts_barrier" ::: "memory");
      }
      __builtin_amdgcn_sched_barrier(0);
      unrolled<2 * F>([&](auto m_) __attribute__((always_inline)) {
        constexpr int m = decltype(m_)::value, f = m / 2, k = m % 2;
        const bf16x8_t x = ring[f % 8];
        if constexpr (f < T::F1) {
          if constexpr (f < 2) mfma_first(s[O][f % 2][k], x, kf[k][0]);
          else mfma_next(s[O][f % 2][k], x, kf[k][f / 2]);
        } else if constexpr (f < T::F2) {
          constexpr int n = f - T::F1;
          if constexpr (n < 2) mfma_first(dp[O][n % 2][k], x, vf[k][0], nd[n % 2]);
          else mfma_next(dp[O][n % 2][k], x, vf[k][n / 2]);
        } else if constexpr (f < T::F3) {
          gt::mfma(dv[f - T::F2][k], x, __builtin_bit_cast(bf16x8_t, p[O][k]));
        } else {
          gt::mfma(dk[f - T::F3][k], x, __builtin_bit_cast(bf16x8_t, e[O][k]));
        }
        // the fragment 7 on, once both products of its place's last one are issued; with three buffers
        // the next tile is known to be there, and the one before done with, only now
        if constexpr (SUB == 0 && BUFS == 3 && m == 2 * F - 13) {
          wait_loads();
          barrier();
        }
        if constexpr (m % 2 == 1) {
          constexpr int n = (m + 13) / 2;
          if constexpr (n < F) read(std::integral_constant<int, n>{}, I0{}, Oth{}, Oth{});
          else read(std::integral_constant<int, n - F>{}, I0{}, Sub{}, I0{});
        } else if constexpr (m >= 2 && (m + 12) / 2 < F) {
          read(std::integral_constant<int, (m + 12) / 2>{}, I1{}, Oth{}, Oth{});
        }
        // P and dS: 64 operations, 16 multiplications and additions with their exponentials,
        // then 16 products with the roundings
        spread<m, 2 * F, 64>([&](auto i_) __attribute__((always_inline)) {
          constexpr int i = decltype(i_)::value;
          constexpr int v = i % 32 / 2, q = v / 8, kk = v / 4 % 2, r = v % 4;
          if constexpr (i < 32) {
            float y = s[SUB][q][kk][r];
            if constexpr (i % 2 == 0) y = fmaf(y, c, -l2[q][r]);
            else y = __builtin_amdgcn_exp2f(y);
            here(y);
            s[SUB][q][kk][r] = y;
            if (i == 31 && mask) {
#pragma unroll
              for (int z = 0; z < 16; ++z) {
                const int zq = z / 8, zk = z / 4 % 2, zr = z % 4;
                const int qq = qpos + SUB * 32 + zq * 16 + 4 * g + zr;
                if ((a.causal && kv0 + 16 * zk + i16 > qq) || (VARLEN && qq >= kend[zk]))
                  s[SUB][zq][zk][zr] = 0.f;
              }
            }
          } else if constexpr (i % 2 == 0) {
            float y = dp[SUB][q][kk][r] * s[SUB][q][kk][r];
            here(y);
            dp[SUB][q][kk][r] = y;
          } else {
            typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
            constexpr int w = v / 2, wq = w / 4, wk = w / 2 % 2, wr = w % 2;
            const auto& from = v % 2 == 0 ? s[SUB][wq][wk] : dp[SUB][wq][wk];
            unsigned y = __builtin_bit_cast(unsigned, bf16x2_t{(__bf16)from[2 * wr], (__bf16)from[2 * wr + 1]});
            here(y);
            (v % 2 == 0 ? p : e)[SUB][wk][wq * 2 + wr] = y;
          }
        });
        // statistics: delta of the rows that are read; log-sum-exp of the next step's P
        if constexpr (m == 4 || m == 6) nd[(m - 4) / 2] = *(stat_ptr)(uintptr_t)(nw + 256 + O * 128 + (m - 4) * 32);
        constexpr int L2 = F + 4;                // all of this step's are used
        if constexpr (m == L2 || m == L2 + 2)
          l2[(m - L2) / 2] = *(stat_ptr)(uintptr_t)((SUB == 0 ? sw : nw) + O * 128 + (m - L2) * 32);
        if constexpr (SUB == 0) {
          // on to the next tile's rows, once this step's are read; and to this one's columns
          constexpr int A = 2 * T::F2 - 8, B = 2 * F - 12;
          if constexpr (m >= A && m - A < DQK / 32) qr[m - A] += by_row;
          if constexpr (m >= A && m - A < DV / 32) orow[m - A] += by_row;
          if constexpr (m == A) nw += by_row;
          if constexpr (m >= B) {
            constexpr int n = m - B;             // 12 slots
            if constexpr (n < DV / 16) oc[n] += by_col;
            if constexpr (n < DQK / 16) qc[n] += by_col;
          }
        } else {
          constexpr int EVERY = 2 * F / LOADS;
          if constexpr (m % EVERY == 4 && m / EVERY < LOADS) load(std::integral_constant<int, m / EVERY>{});
          if (m == 2 * F - 2) load_stats();
          if (m == 2 * F - 3) sw = nw;
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;

    if constexpr (BUFS == 4) wait_loads<LOADS>();     // all but the third tile's
    else wait_loads();
    barrier();
    // S, dP of the first half and the operands of the first step
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      l2[t] = *(stat_ptr)(uintptr_t)(sw + t * 64);
      nd[t] = *(stat_ptr)(uintptr_t)(sw + 256 + t * 64);
    }
    unrolled<T::F2>([&](auto f_) __attribute__((always_inline)) {
      constexpr int f = decltype(f_)::value, n = f - T::F1;
      read(f_, P0{}, P0{}, P0{});
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        if constexpr (f < 2) mfma_first(s[0][f][k], ring[f % 8], kf[k][0]);
        else if constexpr (f < T::F1) mfma_next(s[0][f % 2][k], ring[f % 8], kf[k][f / 2]);
        else if constexpr (n < 2) mfma_first(dp[0][n % 2][k], ring[f % 8], vf[k][0], nd[n % 2]);
        else mfma_next(dp[0][n % 2][k], ring[f % 8], vf[k][n / 2]);
      }
    });
#pragma unroll
    for (int k = 0; k < 2; ++k) p[1][k] = e[1][k] = u32x4_t{0, 0, 0, 0};
    unrolled<7>([&](auto f_) __attribute__((always_inline)) { read(f_, P0{}, P1{}, P0{}); });
    gt::settle();

#pragma unroll 1
    for (int u = 0; u < total; ++u) {
      const bool mask = (a.causal && qpos < kv0 + 31) || (VARLEN && qpos + 63 >= end_w);
      step(P0{}, mask);
      rbuf = rbuf == BUFS - 1 ? 0 : rbuf + 1;
      by_row = rbuf == BUFS - 1 ? -(BUFS - 1) * BUF : BUF;
      step(P1{}, mask);
      to = to == lw + (BUFS - 1) * BUF ? lw : to + BUF;
      advance();
      if (u > 0) cbuf = cbuf == BUFS - 1 ? 0 : cbuf + 1;
      by_col = cbuf == BUFS - 1 ? -(BUFS - 1) * BUF : BUF;
      if (++ch == G) {
        ch = 0;
        qpos -= 64;
      }
    }
    // the last half's gradients
    unrolled<F>([&](auto f_) __attribute__((always_inline)) {
      constexpr int f = decltype(f_)::value;
      if constexpr (f >= T::F2) {
        read(f_, P0{}, P1{}, P1{});
        read(f_, P1{}, P1{}, P1{});
#pragma unroll
        for (int k = 0; k < 2; ++k)
          if constexpr (f < T::F3) gt::mfma(dv[f - T::F2][k], ring[f % 8], __builtin_bit_cast(bf16x8_t, p[1][k]));
          else gt::mfma(dk[f - T::F3][k], ring[f % 8], __builtin_bit_cast(bf16x8_t, e[1][k]));
      }
    });
    wait_loads();
    gt::settle();
    barrier();
  }

  // ---- to memory in whole rows, through 32 rows of LDS per wave
  constexpr int ROWS_LDS = 32 * (DQK > DV ? T::QR : T::OR);
  char* mine = smem + wid * ROWS_LDS;
  const long out = ((long)b * a.Skv + kv0) * a.Hk + kvh;
  auto store = [&](const auto& acc, auto d_, float scale, bf16* dst) __attribute__((always_inline)) {
    constexpr int D = decltype(d_)::value, CH = D / 8;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int t = 0; t < D / 16; ++t) {
        bf16x4_t w;
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = (__bf16)(acc[t][k][r] * scale);
        const int row = k * 16 + i16, ch = (2 * t + (g >> 1)) ^ place(D * 2, row);
        *reinterpret_cast<bf16x4_t*>(mine + row * D * 2 + (ch << 4) + (g & 1) * 8) = w;
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    // a wave reads what it wrote itself
    for (int c = lane; c < 32 * CH; c += 64) {
      const int row = c / CH, ch = c % CH;
      if (kv0 + row < a.Skv)
        *reinterpret_cast<uint4*>(dst + (long)row * a.Hk * D + ch * 8) =
            *reinterpret_cast<const uint4*>(mine + row * D * 2 + ((ch ^ place(D * 2, row)) << 4));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  store(dk, std::integral_constant<int, DQK>{}, a.scale, a.dk + out * DQK);
  store(dv, std::integral_constant<int, DV>{}, 1.f, a.dv + out * DV);
}

}  // namespace fa
}  // namespace amd_ops
