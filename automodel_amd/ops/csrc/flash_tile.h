// Tiles and MFMA fragments of the flash-attention kernels (gfx950).
//
// A tile is [rows][D] bf16 in LDS, rows padded to a power of two (128, 256 or 512
// bytes), filled by direct global->LDS loads of 16 bytes a lane. A wave's load writes
// 1024 consecutive bytes, so the bank swizzle is put into the global side: the 16-byte
// slot s of row r holds the row's chunk s ^ swz(r). swz serves both kinds of read
// without bank conflicts:
//   * read_rows: lane = row, 8 consecutive columns (ds_read_b128; 16 rows at one slot
//     must land in 16 slots: swz takes all values of its bits over 16 rows);
//   * read_cols: lane = column, 8 rows (two ds_read_b64_tr_b16; 4 rows x 4 slots must
//     not meet: the upper bits of swz differ within 4 consecutive rows).
//
// Products are 32x32x16 MFMAs. S[k][q] = K Q^T leaves lane (q = lane & 31, half = lane
// >> 5) with the k rows (r & 3) + 8 (r >> 2) + 4 half, r = 0..15. The next product sums
// over those k, and a sum may run in any order: its other operand is read in the same
// order (read_cols takes rows 4 half + 0..3 and 8 + 4 half + 0..3), so that scores go
// from one MFMA into the next without a shuffle or a trip through LDS.
#pragma once

#include "common.h"
#include "lds_load.h"

namespace amd_ops {
namespace fa {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;

__host__ __device__ constexpr int row_bytes(int d) { return d <= 64 ? 128 : d <= 128 ? 256 : 512; }

template <int D>
__device__ __forceinline__ int swz(int row) {
  if constexpr (row_bytes(D) == 128) return (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
  else return ((row & 3) << 2) | ((row >> 2) & 3);
}

__device__ __forceinline__ f32x16_t mma(bf16x8_t a, bf16x8_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ f32x16_t zero16() {
  f32x16_t z;
#pragma unroll
  for (int r = 0; r < 16; ++r) z[r] = 0.f;
  return z;
}

// row of register r of a 32x32 accumulator
__device__ __forceinline__ int acc_row(int r, int half) { return (r & 3) + 8 * (r >> 2) + 4 * half; }

// 16-byte direct loads of ROWS x D into the tile at LDS address `lds`: rows
// row0.. of a tensor whose rows are `stride` bytes apart, clamped to the last of `left`
// remaining rows and to the first `chunks` 16-byte pieces of a row (callers mask what lies
// beyond).
template <int D, int ROWS, int WAVES>
constexpr int tile_loads() { return ROWS * row_bytes(D) / 1024 / WAVES; }   // per wave

template <int D, int ROWS, int WAVES>
__device__ __forceinline__ void load_tile(const void* base, unsigned stride, int left, unsigned lds,
                                          int chunks = D / 8) {
  constexpr int RB = row_bytes(D), PER = 1024 / RB;     // rows of one wave's load
  constexpr int N = ROWS * RB / 1024;
  static_assert(N % WAVES == 0, "every wave issues the same number of loads");
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slot = lane % (RB / 16);
#pragma unroll
  for (int i = 0; i < N / WAVES; ++i) {
    const int j = i * WAVES + wid;
    const int row = j * PER + lane / (RB / 16);
    int chunk = slot ^ swz<D>(row);
    if (chunk >= chunks) chunk = 0;                     // any valid address
    const unsigned off = (unsigned)min(row, left - 1) * stride + chunk * 16;
    load_lds16(lds + j * 1024, base, off);
  }
}

// per-lane offsets of the reads; `tile32` and `chunk` are compile-time
template <int D>
__device__ __forceinline__ unsigned rows_base() {
  const int lane = threadIdx.x & 63, row = lane & 31, half = lane >> 5;
  return row * row_bytes(D) + ((half ^ swz<D>(row)) << 4);
}
template <int D>
__device__ __forceinline__ unsigned cols_base() {
  const int lane = threadIdx.x & 63, i = lane & 15, half = lane >> 5;
  const int row = 4 * half + (i >> 2), slot = ((lane >> 4) & 1) * 2 + ((i & 3) >> 1);
  return row * row_bytes(D) + ((slot ^ swz<D>(row)) << 4) + (i & 1) * 8;
}

// lane (row = lane & 31, half): columns 16 c + 8 half + 0..7 of row 32 sub + row
template <int D>
__device__ __forceinline__ bf16x8_t read_rows(const char* smem, unsigned tile, unsigned base, int sub,
                                              int c) {
  return *reinterpret_cast<const bf16x8_t*>(smem + tile + (base ^ (c << 5)) + sub * 32 * row_bytes(D));
}

// lane (column = 32 t + (lane & 31), half): rows 16 c + 4 half + {0..3, 8..11} of the
// tile's 32-row part `sub`
template <int D>
__device__ __forceinline__ bf16x8_t read_cols(const char* smem, unsigned tile, unsigned base, int sub,
                                              int c, int t) {
  typedef __attribute__((address_space(3))) bf16x4_t* lds_ptr;
  const char* p = smem + tile + (base ^ (t << 6)) + (sub * 32 + c * 16) * row_bytes(D);
  const char* p8 = smem + tile + (base ^ (t << 6) ^ 32) + (sub * 32 + c * 16 + 8) * row_bytes(D);
  const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_ptr)p);
  const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_ptr)p8);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// the same with rows 16 c + 8 half + 0..7, the order of read_rows' columns, for products of
// a row-read with a column-read tile
template <int D>
__device__ __forceinline__ unsigned cols_base_natural() {
  const int lane = threadIdx.x & 63, i = lane & 15, half = lane >> 5;
  const int row = 8 * half + (i >> 2), slot = ((lane >> 4) & 1) * 2 + ((i & 3) >> 1);
  return row * row_bytes(D) + ((slot ^ swz<D>(row)) << 4) + (i & 1) * 8;
}
template <int D>
__device__ __forceinline__ bf16x8_t read_cols_natural(const char* smem, unsigned tile, unsigned base,
                                                      int c, int t) {
  typedef __attribute__((address_space(3))) bf16x4_t* lds_ptr;
  const char* p = smem + tile + (base ^ (t << 6)) + c * 16 * row_bytes(D);
  const char* p4 = smem + tile + (base ^ (t << 6) ^ 16) + (c * 16 + 4) * row_bytes(D);
  const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_ptr)p);
  const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_ptr)p4);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

// registers 8 c .. 8 c + 7 of an accumulator as the operand of the next product
__device__ __forceinline__ bf16x8_t pack8(const f32x16_t& p, int c) {
  bf16x8_t out;
#pragma unroll
  for (int j = 0; j < 8; ++j) out[j] = (__bf16)p[8 * c + j];
  return out;
}

__device__ __forceinline__ float max_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// a wave's transposed accumulators [D / 32] (column = row of the result), scaled, through
// 32 rows of LDS of its own to whole-row stores of bf16: the first `rows` rows and `chunks`
// 16-byte pieces of a row
template <int D>
__device__ __forceinline__ void store_rows(const f32x16_t (&acc)[D / 32], float scale, char* mine,
                                           bf16* dst, long row_stride, int rows, int chunks = D / 8) {
  constexpr int RB = row_bytes(D), CH = D / 8, PER = 64 / CH;
  const int lane = threadIdx.x & 63, half = lane >> 5, col = lane & 31;
#pragma unroll
  for (int t = 0; t < D / 32; ++t)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      bf16x4_t w;
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = (__bf16)(acc[t][4 * g + j] * scale);
      *reinterpret_cast<bf16x4_t*>(mine + col * RB + (((t * 4 + g) ^ swz<D>(col)) << 4) + half * 8) = w;
    }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    // a wave reads what it wrote itself
  if (lane < PER * CH) {
    const int ch = lane % CH;
    for (int r = lane / CH; r < 32 && r < rows && ch < chunks; r += PER)
      *reinterpret_cast<uint4*>(dst + (long)r * row_stride + ch * 8) =
          *reinterpret_cast<const uint4*>(mine + r * RB + ((ch ^ swz<D>(r)) << 4));
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// Block -> (tile, head, batch). Consecutive blocks go to the 8 XCDs in turn; the
// blocks of one XCD take neighbouring heads (which share K/V, so they stay in its L2),
// longest tiles first, so that the last wave of blocks is made of short ones.
struct Place { int tile, head, batch; };
__device__ __forceinline__ Place place_block(int tiles, int heads, int batches, bool longest_last) {
  const int n = heads * batches, id = blockIdx.x;
  int hb, t;
  if (n % 8 == 0) {
    const int per = n / 8, j = id >> 3;
    t = j / per;
    hb = (id & 7) * per + j % per;
  } else {
    t = id / n;
    hb = id % n;
  }
  return {longest_last ? tiles - 1 - t : t, hb % heads, hb / heads};
}

}  // namespace fa
}  // namespace amd_ops
