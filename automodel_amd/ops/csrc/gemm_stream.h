// y[B, N] = x[B, K] W[N, K]^T for 3 to 16 rows of x: the weights as streams through LDS (gfx950).
//
// Bound by the weights' bytes, which are read once, and by the time until the first of them
// arrive. What a kernel with its loads in registers lost, at 8 rows of x: one load of 16 rows a wave
// in flight, LDS writes between loads and matrix instructions (4096 x 4096 8.2 us, now 7.3; 1024 x
// 8192 10.4 and 7.2), and workgroups of 16, 32 or 64 rows whose number is no multiple of the CUs'
// (5120 x 4096 11.9 and 8.8, 10240 x 14336 52.8 and 44.6: 6.6 TB/s). Of 1850 shapes and numbers of rows,
// 128 x 128 to 151936 x 1024, it takes 0.86 of that kernel's time in the mean, 1.06 at most.
#pragma once

#include "common.h"
#include "lds_load.h"

namespace amd_ops {

typedef __bf16 gemv_bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 gemv_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gemv_f32x4 __attribute__((ext_vector_type(4)));

constexpr int MAX_SEGMENTS = 3;

// What a launch computes: weights [n[s], K] whose blocks begin at first[s]. With a
// gated product, w[0] and w[1] are gate and up and there is one output.
struct Rows {
  const bf16* x;
  const bf16* w[MAX_SEGMENTS];
  bf16* y[MAX_SEGMENTS];
  int n[MAX_SEGMENTS];
  int first[MAX_SEGMENTS];   // INT_MAX: no such segment
  const bf16* bias;          // of a single weight
  float* yf;                 // of a single weight: float32 output instead of y[0]
  const bf16* res;           // of a single weight: added to y
  bool relu2;                // max(y, 0)^2
  int K;
  int group_n;               // > 0: every group_n rows of w take the next B rows of x
  bool stretches;            // skinny: a wave has consecutive tiles of K, else every WAVES-th
};

__device__ __forceinline__ float silu_mul(float g, float u) { return g / (1.f + __expf(-g)) * u; }

// The segment of a block, by selection: an index into the arguments would be one more load
// in the chain that every launch begins with.
struct Segment {
  const bf16* w;
  bf16* y;
  int n, first;
};
__device__ __forceinline__ Segment segment_of(const Rows& p, int block) {
  const bool b1 = block >= p.first[1], b2 = block >= p.first[2];
  return {b2 ? p.w[2] : b1 ? p.w[1] : p.w[0], b2 ? p.y[2] : b1 ? p.y[1] : p.y[0],
          b2 ? p.n[2] : b1 ? p.n[1] : p.n[0], b2 ? p.first[2] : b1 ? p.first[1] : 0};
}

// A workgroup takes R rows of W (GLU: R / 2 of gate and the same of up) and all of x, in XR rows
// of LDS; its waves take consecutive tiles of K each and add up through LDS at the end. A wave has
// a ring of D slots of LDS for itself: 128 columns of its rows of W and x, loaded straight to LDS
// while it multiplies the slots before; no barrier in the loop. x comes from the L2, once for every
// R rows of W: that is why 16 rows of x want more rows of W in a workgroup than 8.
template <int R, int XR, int D, int WAVES, bool GLU>
struct Stream {
  static constexpr int SLOT = (R + XR) * 256;
  static constexpr int LOADS = (R + XR) / 4;      // of a slot: 4 rows each
  static constexpr int RT = (R + 15) / 16;
  static constexpr int OUT = GLU ? R / 2 : R;     // rows of output per workgroup
  static constexpr int RS = 17;
  static constexpr int RED = WAVES * 16 * RT * RS * 4;
  static constexpr int SMEM = WAVES * D * SLOT > RED ? WAVES * D * SLOT : RED;
  static_assert(R % 8 == 0 && (XR == 8 || XR == 16) && D <= 3 && (D - 1) * LOADS < 64);
  static_assert(R + XR >= 16 * RT);   // the last tile's rows beyond R are rows of x, and unused
  static_assert(SMEM <= 160 * 1024);
};

// K % 128 == 0; x and W on 16 bytes; 128 K below 2^32
template <int R, int XR, int D, int WAVES, bool GLU>
__global__ __launch_bounds__(WAVES * WAVE_SIZE) void gemm_stream_kernel(const Rows p, int B) {
  using S = Stream<R, XR, D, WAVES, GLU>;
  extern __shared__ __attribute__((aligned(16))) char stream_lds[];
  const int lane = threadIdx.x & (WAVE_SIZE - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lo16 = lane & 15, hi4 = lane >> 4;
  const Segment seg = segment_of(p, blockIdx.x);
  const int K = p.K, N = seg.n;
  const int n0 = (blockIdx.x - seg.first) * S::OUT;
  const bf16* x = p.x;
  if (p.group_n) x += (long)(n0 / p.group_n) * B * K;   // group_n % OUT == 0

  // Load j covers rows 4j + hi4 of a slot. The 16-byte chunk c of row r lies at c ^ place(r): the
  // 16 lanes that meet in a read, 8 rows' chunk c and the other 8 rows' chunk c ^ 1, hit all banks.
  auto place = [](int r) { return (r & 7) << 1; };
  unsigned off[S::LOADS];
#pragma unroll
  for (int j = 0; j < S::LOADS; ++j) {
    const bool w = j < R / 4;
    const int r = 4 * (w ? j : j - R / 4) + hi4;
    const int row = w ? min(n0 + (GLU ? r % S::OUT : r), N - 1) - n0 : min(r, B - 1);
    off[j] = (unsigned)row * (K * 2u) + (lo16 ^ place(r)) * 16;
  }
  const int tiles = K / 128, per = (tiles + WAVES - 1) / WAVES;
  const int t_lo = wid * per, count = max(min(per, tiles - t_lo), 0);
  // Each workgroup begins elsewhere in its waves' parts of K: rows of W and of x that lie a power of
  // two apart share their memory channels (8 rows of x, 8192 x 8192 21.5 us, 25.0 without).
  int turn = count ? (int)(blockIdx.x % (unsigned)count) : 0;
  const long at0 = (t_lo + turn) * 256l;
  const char* xp = reinterpret_cast<const char*>(x) + at0;
  const char* w0 = reinterpret_cast<const char*>((GLU ? p.w[0] : seg.w) + (long)n0 * K) + at0;
  const char* w1 = GLU ? reinterpret_cast<const char*>(p.w[1] + (long)n0 * K) + at0 : nullptr;

  char* ring = stream_lds + wid * D * S::SLOT;
  const unsigned lds = fa::lds_address(ring);
  auto fetch = [&](unsigned to) {
#pragma unroll
    for (int j = 0; j < S::LOADS; ++j) {
      if (j < R / 4) fa::load_lds16_once(to + j * 1024, GLU && j >= R / 8 ? w1 : w0, off[j]);
      else fa::load_lds16(to + j * 1024, xp, off[j]);
    }
    const long on = (++turn == count ? 1 - count : 1) * 256l;
    w0 += on;
    if (GLU) w1 += on;
    xp += on;
  };

  gemv_f32x4 acc[S::RT];
#pragma unroll
  for (int r = 0; r < S::RT; ++r) acc[r] = gemv_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < D; ++i)
    if (i < count) fetch(lds + i * S::SLOT);
  int slot = 0;
  for (int i = 0; i < count; ++i) {
    const int left = count - 1 - i;               // tiles after this one; up to D - 1 are in flight
    if (D == 1 || left == 0) fa::wait_loads<0>();
    else if (D == 2 || left == 1) fa::wait_loads<S::LOADS>();
    else fa::wait_loads<2 * S::LOADS>();
    const char* at = ring + slot * S::SLOT;
    gemv_bf16x8 xv[4], wv[4][S::RT];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int xr = XR == 8 ? lo16 & 7 : lo16;
      xv[kk] = *reinterpret_cast<const gemv_bf16x8*>(at + (R + xr) * 256 +
                                                     ((kk * 4 + hi4) ^ place(xr)) * 16);
#pragma unroll
      for (int r = 0; r < S::RT; ++r)
        wv[kk][r] = *reinterpret_cast<const gemv_bf16x8*>(at + (r * 16 + lo16) * 256 +
                                                          ((kk * 4 + hi4) ^ place(lo16)) * 16);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    // the slot has been read
    if (left >= D) fetch(lds + slot * S::SLOT);
    slot = slot + 1 == D ? 0 : slot + 1;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int r = 0; r < S::RT; ++r)
        acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[kk][r], xv[kk], acc[r], 0, 0, 0);
  }
  __syncthreads();                                // slots become the reduction buffer
  float* red = reinterpret_cast<float*>(stream_lds);
#pragma unroll
  for (int r = 0; r < S::RT; ++r)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      red[((wid * S::RT + r) * 16 + hi4 * 4 + i) * S::RS + lo16] = acc[r][i];
  __syncthreads();
  auto total = [&](int row, int col) {
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) t += red[(w * 16 * S::RT + row) * S::RS + col];
    return t;
  };
  for (int i = threadIdx.x; i < S::OUT * 16; i += WAVES * WAVE_SIZE) {
    const int row = i % S::OUT, col = i / S::OUT;
    if (n0 + row >= N || col >= B) continue;
    const long o = (long)col * N + n0 + row;
    float t = total(row, col);
    if constexpr (GLU) t = silu_mul(t, total(S::OUT + row, col));
    if (p.relu2) {
      t = fmaxf(t, 0.f);
      t *= t;
    }
    if (p.res) t += bf2f(p.res[o]);
    if (p.yf) p.yf[o] = t;
    else seg.y[o] = f2bf(t);
  }
}

}  // namespace amd_ops
