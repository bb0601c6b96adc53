// What the flash-attention kernels with their instructions in a given order have in common
// (gfx950): MFMAs, code in its place, LDS layout.
#pragma once

#include "flash_tile.h"
#include "gemm_tile.h"

namespace amd_ops {
namespace fa {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

// Products into vector registers, of an operand from LDS and one that stays in AGPRs. The compiler does
// not know what these are (see gt::mfma). Their operands are written by vector instructions at least 16
// MFMAs away. Their results are read by those at least 5 MFMAs of 16 cycles later (the closest is `hide` in
// flash_fwd.h), or after gt::settle.
__device__ __forceinline__ void mfma_first(f32x4_t& d, bf16x8_t a, bf16x8_t b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(d) : "v"(a), "a"(b));
}
__device__ __forceinline__ void mfma_first(f32x4_t& d, bf16x8_t a, bf16x8_t b, f32x4_t c) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %3" : "=&v"(d) : "v"(a), "a"(b), "v"(c));
}
__device__ __forceinline__ void mfma_next(f32x4_t& d, bf16x8_t a, bf16x8_t b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "a"(b));
}

// the same with both operands in vector registers
__device__ __forceinline__ void mfma_first_v(f32x4_t& d, bf16x8_t a, bf16x8_t b, f32x4_t c) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %3" : "=&v"(d) : "v"(a), "v"(b), "v"(c));
}
__device__ __forceinline__ void mfma_next_v(f32x4_t& d, bf16x8_t a, bf16x8_t b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(d) : "v"(a), "v"(b));
}

// the value is formed here, and not where the compiler would rather have it
template <class T>
__device__ __forceinline__ void here(T& x) { asm volatile("" : "+v"(x)); }

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

// The 16-byte slot of a row's chunk c is c ^ place(row): no conflicts between the 32 bytes of 8 rows
// that meet in a read of columns, nor between the 16 lanes that meet in a read of rows, which are
// 8 rows' chunk c and the other 8 rows' chunk c ^ 1 (lanes 0-3, 12-15, 20-27 and so on).
__device__ __forceinline__ int place(int bytes, int row) {
  return bytes % 256 == 0 ? (row & 7) << 1 : (row & 6);
}

}  // namespace fa
}  // namespace amd_ops
