// 256 x 256 tile of a bf16 matrix product with f32 accumulation (gfx950), for four waves.
//
//   out[r, c] = sum_s R(r, s) C(c, s)
//
// C lies in memory with the output index contiguous (COLS: a row per summed index), R so or
// with the summed index contiguous (a row per output row): g^T x and g w take their tensors
// as they are. (x w^T, both with the summed index contiguous, would load two steps of both at a time,
// too late for 128 KB of buffers: 1360 TFLOP/s where the library has 1580.)
//
// A wave computes 128 x 128: 256 accumulators in the AGPRs, one wave a SIMD. Its instructions
// issue in order, so nothing but their order hides them: a step of 32 of the summed index
// is 64 MFMAs of 16 cycles, and every other instruction has its slot behind one of them,
// no two LDS instructions in the same slot (clumps of reads or loads stall the MFMAs: 1260
// against 1720 TFLOP/s with operands of zeros; scalar arithmetic between the steps cost 10%).
// Operands of the next step are read into a second set of registers meanwhile, the step
// after that is in LDS or in flight: direct loads, 128 KB of buffers. 8 groups of about 2048 rows, 4096 x
// 2048: by 64 x 128 wave tiles, two waves a SIMD, 272 (g^T x) and 326 us (g w), so 212 and 260.
// 8192^3: 1530 and 1560 TFLOP/s, 2040 with operands of zeros, 82% of the matrix cores' peak; the
// rest are the barriers and a tile's first loads and stores, 8 us each round.
//
// 16x16x32 MFMAs rather than 32x32x16: the card's power limit binds, and they take less of it
// (of the rate with zeros the former keep 0.85, the latter 0.74 with random numbers).
//
// LDS. COLS: steps of [32][256], 4 of them, read by transposing reads; 16 columns of a row
// are 32 bytes, and these are permuted within a row so that the 8 rows that meet in a read
// lie in 8 different places of 256 bytes. Otherwise two steps together, [256][64], twice: whole
// 128-byte lines are loaded (with 64 bytes per step 1340 against 1490 TFLOP/s, 8192 x 28672 x
// 4096); 16-byte pieces permuted by row for the 16 rows that meet in a read.
#pragma once

#include "common.h"
#include "flash_tile.h"

namespace amd_ops {
namespace gt {

using fa::bf16x4_t;
using fa::bf16x8_t;
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int STEP = 32, TILE = 256, THREADS = 256;
constexpr int HALF = 65536, SMEM = 2 * HALF;     // either operand's buffers: two pairs of steps

// In asm, so that the accumulators stay in AGPRs: left to itself the compiler moved some of
// them to and fro in the loop for small changes of its schedule. The compiler does not
// know what it is: nothing but loads may write its operands shortly before, and
// `settle` comes before the accumulators are read.
__device__ __forceinline__ void mfma(f32x4_t& d, bf16x8_t a, bf16x8_t b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(d) : "v"(a), "v"(b));
}
__device__ __forceinline__ void settle() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

// 16 bytes a lane to the LDS address lds + to
__device__ __forceinline__ void load_lds(unsigned lds, int to, unsigned off, const char* base) {
  fa::load_lds16(lds + to, base, off);
}

// What a block multiplies: pointers to the tile's first row and column and the sum's
// first element. A COLS operand has `after` rows from that one on and `before` rows before it.
struct Tile {
  const bf16 *r, *c;
  const bf16 *r2, *c2;         // a second pair, added to the sum, or null
  long r_ld, c_ld;             // elements from row to row in memory
  int rows, cols;              // of the output, from the tile's first on
  int sum;                     // a multiple of 64 unless both operands are COLS
  int before, after;
};

template <bool COLS>
struct Operand {
  static constexpr int N = COLS ? 4 : 8;       // loads of a wave: for a step, or for a pair
  static constexpr int W = COLS ? 8 : 2;
  unsigned off[N];             // a lane's part of the loads' addresses
  unsigned win[W];             // and of the reads', in the pair of buffers at hand
  const char *base, *second;
  unsigned ld;
  int at, limit;               // position of base in the sum, and the last one

  // edge: rows or columns of the output that are left; half: which 128 of the tile
  __device__ __forceinline__ void init(const bf16* p, const bf16* p2, long ld_, int edge, const Tile& t,
                                       unsigned lds, int wid, int half) {
    const int lane = threadIdx.x & 63, i = lane & 15, g = lane >> 4;
    ld = (unsigned)(ld_ * 2);
    second = reinterpret_cast<const char*>(p2);
    if constexpr (COLS) {
      // the last step ends with the tensor: its first rows are the step's before, or another
      // group's, and are cleared (`clear`). Fewer than 32 rows in all: the last one repeats.
      limit = max(t.after - STEP, -t.before);
      at = min(0, limit);
      base = reinterpret_cast<const char*>(p + at * ld_);
      const int have = min(t.before + t.after, STEP);
#pragma unroll
      for (int h = 0; h < N; ++h) {
        const int row = 8 * h + 2 * wid + (lane >> 5), ch = (lane & 31) ^ (place(row) << 1);
        off[h] = min(row, have - 1) * ld + (ch >= edge / 8 ? 0 : ch * 16);
      }
#pragma unroll
      for (int q = 0; q < W; ++q) {
        const int row = 8 * g + (i >> 2);
        win[q] = lds + row * 512 + ((place(row) ^ q) << 5) + (i & 3) * 8 + half * 256;
      }
    } else {
      limit = t.sum - 2 * STEP;
      at = 0;
      base = reinterpret_cast<const char*>(p);
#pragma unroll
      for (int h = 0; h < N; ++h) {
        const int row = (4 * h + wid) * 8 + (lane >> 3), ch = (lane & 7) ^ ((row >> 1) & 7);
        off[h] = min(row, edge - 1) * ld + ch * 16;
      }
#pragma unroll
      for (int q = 0; q < W; ++q)
        win[q] = lds + i * 128 + (((q * 4 + g) ^ (i >> 1)) << 4) + half * 16384;
    }
  }
  static __device__ __forceinline__ int place(int row) { return (row & 3) | ((row >> 1) & 4); }

  // on by a step or a pair; beyond the last one the second pair of operands, or no further
  __device__ __forceinline__ void seek() {
    if (at == limit && second) {
      base = second;
      second = nullptr;
      at = 0;
    } else {
      const int d = min(limit - at, COLS ? STEP : 2 * STEP);
      at += d;
      base += COLS ? (unsigned long)(unsigned)d * ld : (unsigned long)(unsigned)d * 2;
    }
  }
  // 16 rows or columns q of step P of the pair; part 0 and 1: half of it, 2: all
  template <int P>
  __device__ __forceinline__ void read(bf16x8_t& d, int q, int part) const {
    if constexpr (COLS) {
      typedef __attribute__((address_space(3))) bf16x4_t* lds_ptr;
      const unsigned p = win[q] + P * 16384;
      if (part != 1) {
        const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_ptr)(uintptr_t)p);
        d[0] = lo[0]; d[1] = lo[1]; d[2] = lo[2]; d[3] = lo[3];
      }
      if (part != 0) {
        const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_ptr)(uintptr_t)(p + 4 * 512));
        d[4] = hi[0]; d[5] = hi[1]; d[6] = hi[2]; d[7] = hi[3];
      }
    } else if (part != 1) {
      typedef __attribute__((address_space(3))) bf16x8_t* lds_ptr;
      d = *(lds_ptr)(uintptr_t)(win[P] + q * 2048);
    }
  }
  // after fragment q of a pair's second step the window is moved to the other pair
  __device__ __forceinline__ void move(int q, int by) {
    if constexpr (COLS) win[q] += by;
    else if (q == 7) {
      win[0] += by;
      win[1] += by;
    }
  }
  // rows of step s of a COLS operand that are not of the sum; true if there were any
  __device__ __forceinline__ bool clear(int s, int sum, char* buf) const {
    const int b = min(s * STEP, limit), lo = min(s * STEP - b, STEP);
    const int hi = max(min(sum - b, STEP), lo);
    if (lo == 0 && hi == STEP) return false;
    for (int i = threadIdx.x; i < STEP * 32; i += THREADS)
      if (i / 32 < lo || i / 32 >= hi)
        *reinterpret_cast<uint4*>(buf + (s & 3) * 16384 + i * 16) = uint4{0, 0, 0, 0};
    return true;
  }
};

__device__ __forceinline__ void zero(f32x4_t (&acc)[8][8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
}

// The product into acc[i][j]: rows 16 i + (lane & 15) and columns 16 j + 4 (lane >> 4) + 0..3
// of the wave's 128 x 128 (waves 2 x 2 of the tile).
template <bool RC>
__device__ __forceinline__ void multiply(f32x4_t (&acc)[8][8], const Tile& t, char* smem) {
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned lds = fa::lds_address(smem);
  Operand<RC> R;
  Operand<true> Q;
  R.init(t.r, t.r2, t.r_ld, t.rows, t, lds, wid, wid >> 1);
  Q.init(t.c, t.c2, t.c_ld, t.cols, t, lds + HALF, wid, wid & 1);
  const int steps = (t.sum + 2 * STEP - 1) / (2 * STEP) * 2 * (t.r2 ? 2 : 1);
  const int whole = RC ? t.sum / STEP : steps;    // steps without rows that are not of the sum
  unsigned cur = lds + wid * 1024, oth = cur + HALF / 2;      // pairs of buffers
  int by = HALF / 2;

  // the loads of four steps; where R comes by pairs, of three and of R's second pair
  auto rows = [&](unsigned to, int at) {
#pragma unroll
    for (int h = 0; h < Operand<RC>::N; ++h) load_lds(to, at + h * 4096, R.off[h], R.base);
    R.seek();
  };
  auto cols = [&](unsigned to, int at) {
#pragma unroll
    for (int h = 0; h < 4; ++h) load_lds(to, HALF + at + h * 4096, Q.off[h], Q.base);
    Q.seek();
  };
  rows(cur, 0);
  cols(cur, 0);
  if (RC) rows(cur, 16384);
  cols(cur, 16384);
  if (RC) rows(oth, 0);
  cols(oth, 0);
  rows(oth, RC ? 16384 : 0);
  if (RC) cols(oth, 16384);
  __builtin_amdgcn_sched_barrier(0);
  zero(acc);

  bf16x8_t rf[2][8], cf[2][8];
  // fragments in the order of their use: a row's, all columns', the other rows'
  auto read = [&](auto p_, int f, int part) {
    constexpr int P = decltype(p_)::value;
    if (f == 0 || f >= 9) R.template read<P>(rf[P][f == 0 ? 0 : f - 8], f == 0 ? 0 : f - 8, part);
    else Q.template read<P>(cf[P][f - 1], f - 1, part);
  };
  auto move = [&](int f) {
    if (f == 0 || f >= 9) R.move(f == 0 ? 0 : f - 8, by);
    else Q.move(f - 1, by);
  };
  auto clear = [&](int s) {
    if constexpr (RC) {
      const bool r = R.clear(s, t.sum, smem), q = Q.clear(s, t.sum, smem + HALF);
      if (r || q) fa::barrier();
    }
  };
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  fa::wait_loads<RC ? 24 : 16>();
  fa::barrier();
  if (whole < 1) clear(0);
#pragma unroll
  for (int f = 0; f < 16; ++f) read(P0{}, f, 2);

  // Step P of a pair. Where its loads go to has been read into registers by all waves:
  //   RC:   four loads of either operand, for the step four on
  //   else: P 0: two steps of columns, for three and four on; P 1: rows, for the pair two on
  // and what the reads take has landed: at most those loads are in flight that are later.
  auto step = [&](auto p_, int s) {
    constexpr int P = decltype(p_)::value;
    fa::wait_loads<RC ? 16 : P == 0 ? 12 : 8>();
    fa::barrier();
    if (RC && s + 1 >= whole && s + 1 < steps) clear(s + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < 64; ++m) {
      const int n = m / 8, slot = m % 8;
      mfma(acc[n][slot], cf[P][slot], rf[P][n]);
      if (slot < 4) read(std::integral_constant<int, 1 - P>{}, n * 2 + slot / 2, slot % 2);
      if (P == 0 && slot == 4) {
        move(n * 2);
        move(n * 2 + 1);
      }
      if constexpr (RC) {
        if (slot == 6 && n % 2 == 0) load_lds(cur, P * 16384 + n / 2 * 4096, R.off[n / 2], R.base);
        if (slot == 6 && n % 2 == 1) load_lds(cur, HALF + P * 16384 + n / 2 * 4096, Q.off[n / 2], Q.base);
        if (m == 60) R.seek();
        if (m == 63) Q.seek();
      } else {
        if (slot == 6) {
          if (P == 1) load_lds(cur, n * 4096, R.off[n], R.base);
          else if (n < 4) load_lds(oth, HALF + 16384 + n * 4096, Q.off[n], Q.base);
          else load_lds(cur, HALF + (n - 4) * 4096, Q.off[n - 4], Q.base);
        }
        if (P == 1 && m == 63) R.seek();
        if (P == 0 && (m == 31 || m == 63)) Q.seek();
      }
      if (P == 1 && m == 63) {
        const unsigned u = cur;
        cur = oth;
        oth = u;
        by = -by;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll 1
  for (int s = 0; s < steps; s += 2) {
    step(P0{}, s);
    step(P1{}, s + 1);
  }
  fa::wait_loads();
  settle();
  fa::barrier();               // no load or read of the buffers is under way
}

// acc in bf16 to out (the tile's first element, `ld` from row to row), through 8 KB of LDS
// per wave, in whole rows of 16-byte pieces
__device__ __forceinline__ void store(const f32x4_t (&acc)[8][8], char* smem, bf16* out, long ld, int rows,
                                      int cols) {
  const int lane = threadIdx.x & 63, i16 = lane & 15, g = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  char* mine = smem + wid * 8192;
  const int c0 = (wid & 1) * 128, chunks = min(cols - c0, 128) / 8;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int ch = (2 * j + (g >> 1)) ^ i16;
        bf16x4_t w;
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = (__bf16)acc[p * 2 + i][j][r];
        *reinterpret_cast<bf16x4_t*>(mine + (i * 16 + i16) * 256 + ch * 16 + (g & 1) * 8) = w;
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    // a wave reads what it wrote itself
    const int r0 = (wid >> 1) * 128 + p * 32;
    if (i16 < chunks)
      for (int r = g; r < 32 && r < rows - r0; r += 4)
        *reinterpret_cast<uint4*>(out + (r0 + r) * ld + c0 + i16 * 8) =
            *reinterpret_cast<const uint4*>(mine + r * 256 + ((i16 ^ (r & 15)) << 4));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}

}  // namespace gt
}  // namespace amd_ops
