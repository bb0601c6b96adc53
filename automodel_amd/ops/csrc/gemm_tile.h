// 256 x 256 tiles of bf16 matrix products with f32 accumulation (gfx950), one after another by the four waves
// of a workgroup.
//
//   out[r, c] = sum_s R(r, s) C(c, s)
//
// Either operand lies in memory with the output index contiguous (COLS: a row per summed index) or with the
// summed index contiguous (a row per output row or column): g^T x, g w and x w^T take their tensors as they
// are.
//
// A wave computes 128 x 128: 256 accumulators in the AGPRs, one wave a SIMD. Its instructions issue in order,
// so nothing but their order hides them: a step of 32 of the summed index is 64 MFMAs of 16 cycles, and every
// other instruction has its slot behind one of them, no two LDS instructions in the same slot where that can be
// (clumps of reads or loads stall the MFMAs: 1260 against 1720 TFLOP/s with operands of zeros; scalar
// arithmetic between the steps cost 10%). Operands of the next step are read into a second set of registers
// meanwhile, the steps after that are in LDS or in flight: direct loads, 128 KB of buffers.
//
// 16x16x32 MFMAs rather than 32x32x16: the card's power limit binds, and they take less of it (of the rate with
// zeros the former keep 0.85, the latter 0.74 with random numbers).
//
// One workgroup a CU stays for all its tiles, because a tile of its own workgroup spent 10 us on other things
// than its products, most of it with nothing in flight: 1 to find out what it is, 5.4 until all CUs' first 128
// KB have come at once, 3 for its stores. Here the loads of a tile's last two pairs of steps are the next
// tile's first ones, so that they come during the products and the stores, and a store is only waited for two
// steps into the next tile. g^T x, 128 groups of 512 rows, 768 x 2048: 20.5 -> 16 us a tile.
//
// A tile has 32 NR rows, NR = 4 to 8: with rows it has not got it takes no time. (Groups of 282 rows: two tiles
// of 160 take 10/16 of two of 256.)
//
// LDS. COLS: steps of [32][256], 4 of them, read by transposing reads; 16 columns of a row are 32 bytes, and
// these are permuted within a row so that the 8 rows that meet in a read lie in 8 different places of 256
// bytes. Otherwise two steps together, [256][64], twice: whole 128-byte lines are loaded (with 64 bytes per
// step 1340 against 1490 TFLOP/s, 8192 x 28672 x 4096); 16-byte pieces permuted by row for the 16 rows that
// meet in a read. Where both are loaded so (x w^T), a pair's place is filled again as soon as its second step
// is in registers, a third of a step after that began: there a barrier, and from there on the loads, evenly over what
// is left of the pair. They are waited for in the middle of the next pair's second step. The even spread is worth more
// than a late wait: all loads in the two thirds of a step after the barrier 1406 us, over twice as much 1303, to the
// pair's end 1282 (8192 rows, 4096 -> 28672; of zeros, where the card's power is not the bound, 1302, 1142, 1042).
#pragma once

#include <algorithm>
#include <utility>

#include "common.h"
#include "flash_tile.h"

namespace amd_ops {
namespace fa {

// f(FROM), ..., f(FROM + N - 1) with compile-time arguments
template <int FROM, class F, int... I>
__device__ __forceinline__ void unrolled_(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, FROM + I>{}), ...);
}
template <int N, int FROM = 0, class F>
__device__ __forceinline__ void unrolled(F&& f) {
  unrolled_<FROM>(f, std::make_integer_sequence<int, N>{});
}

// OPS operations spread over SLOTS slots, operation i in slot i SLOTS / OPS: f(i) for those of slot M. (Only
// these are expanded: a test of each operation in each slot took three quarters of the compile time.)
template <int M, int SLOTS, int OPS, class F>
__device__ __forceinline__ void spread(F&& f) {
  constexpr int from = (M * OPS + SLOTS - 1) / SLOTS, to = ((M + 1) * OPS + SLOTS - 1) / SLOTS;
  constexpr int first = from < OPS ? from : OPS, end = to < OPS ? to : OPS;
  unrolled<end - first, first>(f);
}

}  // namespace fa

namespace gt {

using fa::bf16x4_t;
using fa::bf16x8_t;
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));

constexpr int STEP = 32, TILE = 256, THREADS = 256;
constexpr int HALF = 65536;                      // either operand's buffers: two pairs of steps
constexpr int STAGE = 2 * HALF;                  // 4 KB a wave: outputs on their way to memory
constexpr int SMEM = STAGE + 4 * 4096;

// In asm, so that the accumulators stay in AGPRs: left to itself the compiler moved some of
// them to and fro in the loop for small changes of its schedule. The compiler does not
// know what it is: nothing but loads may write its operands shortly before, and
// `settle` comes before the accumulators are read.
__device__ __forceinline__ void mfma(f32x4_t& d, bf16x8_t a, bf16x8_t b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(d) : "v"(a), "v"(b));
}
__device__ __forceinline__ void mfma_first(f32x4_t& d, bf16x8_t a, bf16x8_t b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(d) : "v"(a), "v"(b));
}
__device__ __forceinline__ void settle() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

// 16 bytes a lane to the LDS address lds + to
__device__ __forceinline__ void load_lds(unsigned lds, int to, unsigned off, const char* base) {
  fa::load_lds16(lds + to, base, off);
}
// the same within `num` bytes from the base on; beyond them zeros
__device__ __forceinline__ void load_lds(unsigned lds, int to, unsigned off, const char* base, unsigned num) {
  const unsigned long p = (unsigned long)base;
  const i32x4_t rsrc{(int)(unsigned)p, (int)(unsigned)(p >> 32), (int)num, 0x00027000};
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :: "s"(lds + to), "v"(off), "s"(rsrc) : "memory", "m0");
}

// the same from off + more on, which takes a register for the moment only
__device__ __forceinline__ void load_lds(unsigned lds, int to, unsigned off, unsigned more, const char* base, unsigned num) {
  const unsigned long p = (unsigned long)base;
  const i32x4_t rsrc{(int)(unsigned)p, (int)(unsigned)(p >> 32), (int)num, 0x00027000};
  unsigned at;
  asm volatile("s_mov_b32 m0, %1\n\tv_add_u32 %0, %3, %2\n\tbuffer_load_dwordx4 %0, %4, 0 offen lds"
               : "=&v"(at) : "s"(lds + to), "v"(off), "s"(more), "s"(rsrc) : "memory", "m0");
}

// max(x, 0)^2; NaN stays
__device__ __forceinline__ float relu2(float x) {
  const float y = x < 0.f ? 0.f : x;
  return y * y;
}

// silu(a) b as swiglu.hip has it, to the bit but for quotients below 2^-126: one step of Newton's method instead of a
// division of ten instructions (its quotient is the rounded one but for divisors of 24 ones)
__device__ __forceinline__ float rounded_glu(__bf16 one, __bf16 other) {
  const float a = (float)one, d = 1.f + __expf(-a), r = __builtin_amdgcn_rcpf(d);
  const float sigmoid = d > 3.4e38f ? 0.f : fmaf(fmaf(-d, r, 1.f), r, r);
  return a * sigmoid * (float)other;
}

// the lane, formed anew: what follows from it is not kept in registers over the whole kernel
__device__ __forceinline__ int lane_here() {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));
  return lane;
}

// What is multiplied: pointers to the tile's first row and column and the sum's first element.
struct Tile {
  const bf16 *r = nullptr, *c = nullptr;
  const bf16* up = nullptr;    // GLU: the second matrix of columns
  bf16 *one = nullptr, *other = nullptr;       // KEEP: where its sums go
  const bf16 *r2 = nullptr, *c2 = nullptr;     // a second pair, added to the sum, or null
  int rank = 0, rank_c = 0;    // EXTRA: how long a row of r2 is, a multiple of 32, and of c2, one of 8: zeros behind it
  int rows = 0, cols = 0;      // of the output, from the tile's first on
  int sum = 0;                 // a multiple of 64 unless both operands are COLS
  bf16* out = nullptr;
  float* part = nullptr;       // PARTS: where the tile's sums go instead

  // Member by member: a copy of the whole went through memory, and the wait for it was one for all loads under way (of
  // groups 4% of the time).
  __device__ __forceinline__ Tile() {}
  __device__ __forceinline__ Tile(const Tile& t) { *this = t; }
  __device__ __forceinline__ Tile& operator=(const Tile& t) {
    r = t.r, c = t.c, up = t.up, one = t.one, other = t.other, r2 = t.r2, c2 = t.c2, rank = t.rank, rank_c = t.rank_c;
    rows = t.rows, cols = t.cols, sum = t.sum, out = t.out, part = t.part;
    return *this;
  }
};

// 16 rows how often a wave has, in a tile with so many rows left
__host__ __device__ constexpr int rows16(int rows) { return rows > 224 ? 8 : rows > 128 ? (rows + 31) / 32 : 4; }

// bytes from row to row, below 2^24: a tile's addresses are 32 bits
struct Shape {
  unsigned r, c, out;
};

// SHORT: the sum may end within what is loaded. TWO: 16 rows of one matrix, 16 of the other, 128 of each; the first two
// waves load the one's, the others the other's.
// FEW: one register for the loads' addresses, which are equally far apart, instead of N.
template <bool COLS, bool SHORT, bool TWO = false, bool FEW = false>
struct Operand {
  static_assert(!COLS || !FEW);
  static constexpr int N = COLS ? 4 : 8;       // loads of a wave: for a step, or for a pair
  static constexpr int W = COLS ? 8 : 2;
  unsigned off[FEW ? 1 : N];   // a lane's part of the loads' addresses
  unsigned win[W];             // and of the reads', in the pair of buffers at hand
  const char* base;
  unsigned ld, num;            // bytes: from row to row, and from base on that may be read
  unsigned all;                // COLS: of a row before base; else of the tile's rows
  int left;                    // of the sum

  __device__ __forceinline__ void init(unsigned ld_, int wid) {
    const int lane = threadIdx.x & 63;
    ld = ld_;
#pragma unroll
    for (int h = 0; h < (FEW ? 1 : N); ++h) {
      if constexpr (COLS) {
        const int row = 8 * h + 2 * wid + (lane >> 5);
        off[h] = row * ld + ((lane & 31) ^ (place(row) << 1)) * 16;
      } else {
        const int row = (4 * h + wid) * 8 + (lane >> 3), from = TWO ? h * 16 + (row & 15) : row;
        off[h] = from * ld + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
      }
    }
  }
  // load h, to `to` + `at`
  __device__ __forceinline__ void load(unsigned to, int at, int h) const {
    if constexpr (FEW) load_lds(to, at, off[0], h * (TWO ? 16 : 32) * ld, base, num);
    else load_lds(to, at, off[h], base, num);
  }
  // The loads go on with another tile, `edge` rows or columns of the output wide. What lies outside of it or of
  // the sum is not read: rows beyond are zeros, and so are those of the summed index. (Columns beyond are the
  // next row's; nothing is made of them.)
  __device__ __forceinline__ void aim(const bf16* p, int edge, int sum) {
    base = reinterpret_cast<const char*>(p);
    left = sum;
    all = COLS ? ld - 2 * edge : min(edge, TWO ? TILE / 2 : TILE) * ld;
    count();
  }
  __device__ __forceinline__ void count() {
    if constexpr (COLS) {
      const int n = (SHORT ? min(left, STEP) : STEP) * (int)ld - (int)all;      // the last row ends where the tensor may end
      num = SHORT ? max(n, 0) : n;
    } else {
      num = !SHORT || left > 0 ? all : 0;
    }
  }
  __device__ __forceinline__ void seek() {
    base += COLS ? (unsigned long)(STEP * ld) : (unsigned long)(4 * STEP);
    if constexpr (SHORT) {
      left -= COLS ? STEP : 2 * STEP;
      count();
    }
  }

  // windows on the pair of buffers at `lds`; first: 16 rows or columns that are fragment 0
  __device__ __forceinline__ void look(unsigned lds, int first) {
    const int lane = lane_here(), i = lane & 15, g = lane >> 4;
#pragma unroll
    for (int q = 0; q < W; ++q) {
      if constexpr (COLS) {
        const int row = 8 * g + (i >> 2);
        win[q] = lds + row * 512 + (((first + q) ^ place(row)) << 5) + (i & 3) * 8;
      } else {
        win[q] = lds + (first * 16 + i) * 128 + (((q * 4 + g) ^ (i >> 1)) << 4);
      }
    }
  }
  static __device__ __forceinline__ int place(int row) { return (row & 3) | ((row >> 1) & 4); }

  // fragment q, 16 rows or columns, of step P of the pair; part 0 and 1: half of it, 2: all
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
    } else {
      typedef __attribute__((address_space(3))) bf16x8_t* lds_ptr;
      d = *(lds_ptr)(uintptr_t)(win[P] + q * 2048);
    }
  }
  // after fragment q, of `last` + 1, of a pair's second step its window is moved to the other pair
  __device__ __forceinline__ void move(int q, int last, int by) {
    if constexpr (COLS) {
      win[q] += by;
    } else if (q == last) {
      win[0] += by;
      win[1] += by;
    }
  }
};

// All tiles of a workgroup. SHORT: sums that are no multiple of a pair of steps, or a single pair. Tiles:
// first() and next() are their numbers, or negative; get(number) is the tile; loaded() is called once, while
// the first tile's operands come.
// PARTS: tiles of sums that are added up later, 32 bits in the order of the accumulators.
// RELU2: the results are max(sum, 0)^2.
// GLU: the columns are 16 of one matrix and 16 of another, in turn, so that a lane has the sums of both for its column;
// the results, half as many, are silu(one) other. KEEP: both sums are written too, and silu is of what is
// written.
// EXTRA: the second pair is [rows][rank] and [columns][rank_c], short rows that are loaded as fragments behind the
// sum. They come from the L2, and with them the wave waits for the next tile's loads (8192 rows, a sum of 4096,
// 4096 columns: 192 us without, 190 with it).
template <bool RC, bool CC, class Tiles, bool SHORT = RC && CC, bool PARTS = false, bool EXTRA = false, bool RELU2 = false, bool GLU = false,
          bool KEEP = false>
struct Run {
  static constexpr bool TN = RC && CC, NN = !RC && CC, NT = !CC;
  Tiles& tiles;
  char* smem;
  const Shape shape;
  unsigned lds, cur, oth;      // buffers' addresses: of the pair at hand, of the other
  int by, wid;
  Operand<RC, SHORT, false, KEEP> R;   // (KEEP: with a register for each load others went to memory in every step)
  Operand<CC, SHORT, GLU, KEEP> C;

  __device__ __forceinline__ Run(Tiles& t, const Shape& sh, char* s) : tiles(t), smem(s), shape(sh) {
    wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lds = fa::lds_address(smem);
    cur = lds + wid * 1024;
    oth = cur + HALF / 2;
    by = HALF / 2;
    R.init(shape.r, wid);
    C.init(shape.c, wid);
  }

  // where the loads go on: at a tile, at its second pair of operands before pair `at` + 2, or at the next tile
  __device__ __forceinline__ void aim(const Tile& t) {
    R.aim(t.r, t.rows, t.sum);
    C.aim(GLU && wid >> 1 ? t.up : t.c, t.cols, t.sum);
  }
  __device__ __forceinline__ void go_on(const Tile& t, const Tile& u, int n, int& at) {
    if (NN && !EXTRA && t.r2 && at != n - 2) {
      R.aim(t.r2, t.rows, t.sum);
      C.aim(t.c2, t.cols, t.sum);
      at = n - 2;
    } else {
      aim(u);
    }
  }
  __device__ __forceinline__ void rows(unsigned to, int at) {
#pragma unroll
    for (int h = 0; h < decltype(R)::N; ++h) R.load(to, at + h * 4096, h);
    R.seek();
  }
  __device__ __forceinline__ void cols(unsigned to, int at) {
#pragma unroll
    for (int h = 0; h < decltype(C)::N; ++h) C.load(to, HALF + at + h * 4096, h);
    C.seek();
  }

  // tile t by waves of 16 NR rows, and the loads of the beginning of tile u
  template <int NR>
  __device__ __forceinline__ void tile(const Tile& t, const Tile& u) {
    // pairs of steps; two at least of either pair of operands, as many as are loaded ahead: what is beyond the
    // sum is zeros
    const int n1 = max((t.sum + 2 * STEP - 1) / (2 * STEP), 2), n = NN && !EXTRA && t.r2 ? 2 * n1 : n1;
    f32x4_t acc[NR][8];
    bf16x8_t rf[2][NR], cf[2][8];
    const unsigned pair = lds + (by > 0 ? 0 : HALF / 2);
    R.look(pair, (wid >> 1) * NR);
    C.look(pair + HALF, (wid & 1) * 8);

    // fragments in the order of their use: a row's, all columns', the other rows'
    auto frag = [&](auto p_, int f, int part) __attribute__((always_inline)) {
      constexpr int P = decltype(p_)::value;
      if (f == 0 || f >= 9) R.template read<P>(rf[P][f == 0 ? 0 : f - 8], f == 0 ? 0 : f - 8, part);
      else C.template read<P>(cf[P][f - 1], f - 1, part);
    };
    auto move = [&](int f) __attribute__((always_inline)) {
      if (f == 0 || f >= 9) R.move(f == 0 ? 0 : f - 8, NR - 1, by);
      else C.move(f - 1, 7, by);
    };
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int f = 0; f < 8 + NR; ++f) frag(P0{}, f, 2);

    // Step P of a pair. Loads of the buffers' next contents, in this order:
    //   TN: four of rows and four of columns, for the step four on
    //   NN: P 0: four of columns, for the step four on; P 1: eight of rows, for the pair two on, and four of columns
    //   NT: from P 0 on, when the rows' and columns' fragments are read (MID): eight of both, for the pair two on
    // Waits: what is read next has landed. So many loads are later (NT: of the 16 those before the middle of P 1), and
    // in a tile's first pair the last tile's stores are, 16 at least, of GLU 8 (loads and stores are counted in the order of
    // their issue).
    constexpr int RR = RC ? 2 : 1, CR = CC ? 2 : 1, READS = NR * RR + 8 * CR, S = NR * 8;
    auto step = [&](auto p_, auto first_) __attribute__((always_inline)) {
      constexpr int P = decltype(p_)::value;
      constexpr bool FIRST = decltype(first_)::value;
      constexpr int DENSE = READS > 3 * S / 8 ? READS : 3 * S / 8;
      constexpr int MID = DENSE + 4, OVER = 2 * S - MID;       // NT: slots of a pair that loads are spread over
      constexpr int LATER = (NT ? ((S + S / 2 - MID) * 16 + OVER - 1) / OVER : NN && P == 1 ? 8 : 16) + (FIRST ? (GLU && !KEEP ? 8 : 16) : 0);
      // slots of the reads
      constexpr int FROM = NT && P == 1 ? S / 2 : 0, TO = TN || NN || P == 1 ? S : DENSE;
      if constexpr (!NT) {
        fa::wait_loads<LATER>();
        fa::barrier();
      }
      __builtin_amdgcn_sched_barrier(0);
      fa::unrolled<S>([&](auto m_) __attribute__((always_inline)) {
        constexpr int m = decltype(m_)::value, i = m / 8, j = m % 8;
        if constexpr (NT && P == 0 && m == MID) fa::barrier();
        if constexpr (NT && P == 1 && m == FROM) {
          fa::wait_loads<LATER>();
          fa::barrier();
        }
        if constexpr (FIRST && P == 0) mfma_first(acc[i][j], cf[P][j], rf[P][i]);
        else mfma(acc[i][j], cf[P][j], rf[P][i]);
        if constexpr (m >= FROM && m < TO)
          fa::spread<m - FROM, TO - FROM, READS>([&](auto d_) __attribute__((always_inline)) {
            constexpr int d = decltype(d_)::value;
            // a row's, all columns', the other rows'
            constexpr int D = d - RR - 8 * CR, f = d < RR ? 0 : D < 0 ? 1 + (d - RR) / CR : 9 + D / RR;
            constexpr int each = d < RR || D >= 0 ? RR : CR, part = each == 1 ? 2 : (d < RR ? d : D < 0 ? d - RR : D) % each;
            frag(std::integral_constant<int, 1 - P>{}, f, part);
            if constexpr (P == 0 && part > 0) move(f);
          });
        if constexpr (NT) {
          if constexpr (P * S + m >= MID)
            fa::spread<P * S + m - MID, OVER, 16>([&](auto l_) __attribute__((always_inline)) {
              constexpr int l = decltype(l_)::value / 2, odd = decltype(l_)::value % 2;
              if constexpr (odd) R.load(cur, l * 4096, l);
              else C.load(cur, HALF + l * 4096, l);
              if constexpr (l == 7 && odd) R.seek();
              if constexpr (l == 7 && !odd) C.seek();
            });
        } else if constexpr (TN) {
          fa::spread<m, S, 8>([&](auto l_) __attribute__((always_inline)) {
            constexpr int l = decltype(l_)::value / 2, odd = decltype(l_)::value % 2;
            if constexpr (odd) load_lds(cur, P * 16384 + l * 4096, R.off[l], R.base, R.num);
            else load_lds(cur, HALF + P * 16384 + l * 4096, C.off[l], C.base, C.num);
            if constexpr (l == 3 && odd) R.seek();
            if constexpr (l == 3 && !odd) C.seek();
          });
        } else {
          fa::spread<m, S, P == 0 ? 4 : 12>([&](auto l_) __attribute__((always_inline)) {
            constexpr int l = decltype(l_)::value, q = P == 0 ? l : l - 8;
            if constexpr (q < 0) {
              load_lds(cur, l * 4096, R.off[l], R.base, R.num);
              if constexpr (l == 7) R.seek();
            } else {
              load_lds(cur, HALF + P * 16384 + q * 4096, C.off[q], C.base, C.num);
              if constexpr (q == 3) C.seek();
            }
          });
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      if (P == 1) {
        const unsigned v = cur;
        cur = oth;
        oth = v;
        by = -by;
      }
    };
    using T = std::true_type;
    using F = std::false_type;
    int at = n1 - 2;
    if (at == 0) go_on(t, u, n, at);
    step(P0{}, T{});
    step(P1{}, T{});
#pragma unroll 1
    for (int p = 1; p < n; ++p) {
      if (p == at) go_on(t, u, n, at);
      step(P0{}, F{});
      step(P1{}, F{});
    }
    if constexpr (EXTRA) extra<NR>(acc, t);
    settle();
    if constexpr (PARTS) keep<NR>(acc, t);
    else if constexpr (GLU) store_glu<NR>(acc, t);
    else store<NR>(acc, t);
  }

  template <int NR>
  __device__ __forceinline__ void extra(f32x4_t (&acc)[NR][8], const Tile& t) {
    if (!t.r2) return;
    const int lane = lane_here(), i16 = lane & 15, g = lane >> 4;
    const int r0 = (wid >> 1) * (NR * 16) + i16, c0 = (wid & 1) * 128 + i16;
    const bf16 *r2 = t.r2 + g * 8, *c2 = t.c2 + g * 8;
#pragma unroll 1
    for (int k = 0; k < t.rank; k += 32) {
      bf16x8_t rx[NR], cx[8];          // (rows and columns beyond the edge are loaded again, and not stored)
#pragma unroll
      for (int i = 0; i < NR; ++i)
        rx[i] = *reinterpret_cast<const bf16x8_t*>(r2 + min(r0 + i * 16, t.rows - 1) * t.rank + k);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        cx[j] = k + g * 8 < t.rank_c ? *reinterpret_cast<const bf16x8_t*>(c2 + min(c0 + j * 16, t.cols - 1) * t.rank_c + k)
                                     : bf16x8_t{};
#pragma unroll
      for (int i = 0; i < NR; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) mfma(acc[i][j], cx[j], rx[i]);
    }
  }

  // accumulators to memory as they lie: [wave][i][j][lane], 16 bytes a lane
  template <int NR>
  __device__ __forceinline__ void keep(const f32x4_t (&acc)[NR][8], const Tile& t) {
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(t.part, 0, TILE * TILE * 4, 0x00027000);
    const unsigned at = wid * (NR * 8 * 1024) + lane_here() * 16;
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc[i][j]), rsrc,
                                               at + (i * 8 + j) * 1024, 0, 0);
    asm volatile("" ::: "memory");
  }

  // acc[i][j] in bf16 to memory: rows 16 i + (lane & 15) and columns 16 j + 4 (lane >> 4) + 0..3 of the wave's
  // part, through 4 KB of LDS, in whole rows of 16-byte pieces. No waits: a wave's LDS instructions are carried
  // out in order. Always 4 NR stores, which are counted on (`step`): what is not of the output is out of the
  // buffer's bounds.
  template <int NR>
  __device__ __forceinline__ void store(const f32x4_t (&acc)[NR][8], const Tile& t) {
    const int lane = lane_here(), i16 = lane & 15, g = lane >> 4;
    char* mine = smem + STAGE + wid * 4096;
    const int c0 = (wid & 1) * 128, chunks = min(t.cols - c0, 128) / 8, r0 = (wid >> 1) * (NR * 16);
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(t.out, 0, 0xffffff00, 0x00027000);
    auto put = [&](auto i_) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        bf16x4_t w;
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = (__bf16)(RELU2 ? relu2(acc[decltype(i_)::value][j][r]) : acc[decltype(i_)::value][j][r]);
        *reinterpret_cast<bf16x4_t*>(mine + i16 * 256 + (((2 * j + (g >> 1)) ^ i16) << 4) + (g & 1) * 8) = w;
      }
      asm volatile("" ::: "memory");
    };
    put(std::integral_constant<int, 0>{});
    fa::unrolled<NR>([&](auto i_) __attribute__((always_inline)) {
      constexpr int i = decltype(i_)::value;
      u32x4_t v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k)
        v[k] = *reinterpret_cast<const u32x4_t*>(mine + (4 * k + g) * 256 + ((i16 ^ (4 * k + g)) << 4));
      asm volatile("" ::: "memory");
      if constexpr (i + 1 < NR) put(std::integral_constant<int, i + 1>{});
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int row = r0 + i * 16 + 4 * k + g;
        const unsigned o = row * shape.out + (c0 + i16 * 8) * 2;
        __builtin_amdgcn_raw_buffer_store_b128(v[k], rsrc, row < t.rows && i16 < chunks ? o : 0xfffffff0u, 0, 0);
      }
    });
    asm volatile("" ::: "memory");
  }

  // The same of silu(acc[i][2 j]) acc[i][2 j + 1], 64 columns a wave: 2 NR stores. KEEP: of the sums too, 6 NR.
  template <int NR>
  __device__ __forceinline__ void store_glu(const f32x4_t (&acc)[NR][8], const Tile& t) {
    const int lane = lane_here(), i16 = lane & 15, g = lane >> 4;
    char* mine = smem + STAGE + wid * 4096;
    const int c0 = (wid & 1) * 64, chunks = min(t.cols - c0, 64) / 8, r0 = (wid >> 1) * (NR * 16);
    constexpr int W = KEEP ? 3 : 1;              // what is written of each row
    const auto rsrc = [&](int what) __attribute__((always_inline)) {
      return __builtin_amdgcn_make_buffer_rsrc(what == 0 ? t.out : what == 1 ? t.one : t.other, 0, 0xffffff00, 0x00027000);
    };
    auto put = [&](auto s_) __attribute__((always_inline)) {
      constexpr int i = decltype(s_)::value / W, what = decltype(s_)::value % W;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        bf16x4_t w;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float a = acc[i][2 * j][r], b = acc[i][2 * j + 1][r];
          if constexpr (KEEP) w[r] = (__bf16)(what == 0 ? rounded_glu((__bf16)a, (__bf16)b) : what == 1 ? a : b);
          else w[r] = (__bf16)(a * __builtin_amdgcn_rcpf(1.f + __expf(-a)) * b);
        }
        *reinterpret_cast<bf16x4_t*>(mine + i16 * 128 + (((2 * j + (g >> 1)) ^ (i16 >> 1)) << 4) + (g & 1) * 8) = w;
      }
      asm volatile("" ::: "memory");
    };
    put(std::integral_constant<int, 0>{});
    fa::unrolled<NR * W>([&](auto s_) __attribute__((always_inline)) {
      constexpr int s = decltype(s_)::value, i = s / W;
      u32x4_t v[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int row = 8 * k + (lane >> 3);
        v[k] = *reinterpret_cast<const u32x4_t*>(mine + row * 128 + (((lane & 7) ^ (row >> 1)) << 4));
      }
      asm volatile("" ::: "memory");
      if constexpr (s + 1 < NR * W) put(std::integral_constant<int, s + 1>{});
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int row = r0 + i * 16 + 8 * k + (lane >> 3);
        const unsigned o = row * shape.out + (c0 + (lane & 7) * 8) * 2;
        __builtin_amdgcn_raw_buffer_store_b128(v[k], rsrc(s % W), row < t.rows && (lane & 7) < chunks ? o : 0xfffffff0u, 0, 0);
      }
    });
    asm volatile("" ::: "memory");
  }

  __device__ __forceinline__ void operator()() {
    int id = tiles.first();
    if (id < 0) return;
    Tile t = tiles.get(id);
    aim(t);
    rows(cur, 0);
    cols(cur, 0);
    if (RC) rows(cur, 16384);
    if (CC) cols(cur, 16384);
    rows(oth, 0);
    cols(oth, 0);
    if (RC) rows(oth, 16384);
    if (CC) cols(oth, 16384);
    tiles.loaded();
    fa::wait_loads();
    fa::barrier();
    for (;;) {
      const int next = tiles.next();
      Tile u = t;              // (behind the last one nothing is made of the loads)
      if (next >= 0) u = tiles.get(next);
      switch (rows16(t.rows)) {
        case 8: tile<8>(t, u); break;
        case 7: tile<7>(t, u); break;
        case 6: tile<6>(t, u); break;
        case 5: tile<5>(t, u); break;
        default: tile<4>(t, u); break;
      }
      if (next < 0) break;
      t = u;
    }
    fa::wait_loads();          // no load is under way into LDS that is another workgroup's
    fa::barrier();
  }
};

// one a CU, as many on each of the 8 XCDs
inline long workgroups() {
  static const long n = [] {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      cus = 256;
    return std::min(std::max(cus / 8 * 8, 8), 256);
  }();
  return n;
}

}  // namespace gt
}  // namespace amd_ops
