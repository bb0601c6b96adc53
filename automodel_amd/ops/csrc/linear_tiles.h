// Tiles of y = x w^T and its gradients (linear_grad.hip, linear_out.hip, lora_grad.hip): their order, and how they
// and their sums are cut.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"
#include "gemm_tile.h"

namespace amd_ops {
namespace lg {

enum Form { Y, DX, DW, GLU };

struct Args {
  const bf16 *r, *c;
  bf16* out;
  float* part;                         // [part][tile][height][256], in the order of the accumulators
  int rows, cols, sum;
  int height, parts, per;              // rows of a tile; parts of the sum, and how much of it each but the last has
  const bf16 *r2, *c2;                 // EXTRA: [rows][rank] and [cols][rank_c], whose product is added
  int rank, rank_c;
  bool relu2;                          // Y: max(sum, 0)^2
  const bf16* up;                      // GLU: c is [cols / 2][sum], and so is this
};

// The tiles' order is down 4 row tiles, then on to the next column tile: the 32 tiles of an XCD at a time read
// 4 row tiles and 8 column tiles.
constexpr int DOWN = 4;

__device__ __forceinline__ void place(int i, int nr, int nc, int height, int& r0, int& c0) {
  const int group = i / (DOWN * nc), in = i % (DOWN * nc), down = min(DOWN, nr - group * DOWN);
  r0 = (group * DOWN + in % down) * height;
  c0 = in / down * gt::TILE;
}

// Blocks are dealt to the 8 XCDs in contiguous stretches of the tile list, one part after another.
template <Form F, bool EXTRA = false>
struct Tiles {
  const Args& a;
  const int nc, nr, stride;
  int id, end;
  __device__ __forceinline__ Tiles(const Args& a_)
      : a(a_), nc((a.cols + gt::TILE - 1) / gt::TILE), nr((a.rows + a.height - 1) / a.height), stride(gridDim.x >> 3) {
    const int total = nr * nc * a.parts, per = (total + 7) / 8, x = blockIdx.x & 7;
    id = x * per + (blockIdx.x >> 3);
    end = min((x + 1) * per, total);
  }
  __device__ __forceinline__ int first() const { return id < end ? id : -1; }
  __device__ __forceinline__ int next() {
    id += stride;
    return first();
  }
  __device__ __forceinline__ void loaded() const {}
  __device__ __forceinline__ gt::Tile get(int u) const {
    const int s = u / (nr * nc), from = s * a.per;
    int r0, c0;
    place(u - s * nr * nc, nr, nc, a.height, r0, c0);
    gt::Tile t;
    t.rows = min(a.rows - r0, a.height);
    t.cols = a.cols - c0;
    t.sum = min(a.sum - from, a.per);
    t.r = F == DW ? a.r + (long)from * a.rows + r0 : a.r + (long)r0 * a.sum + from;
    t.c = F == Y ? a.c + (long)c0 * a.sum + from : a.c + (long)from * a.cols + c0;
    t.out = a.out + (long)r0 * a.cols + c0;
    if constexpr (F == GLU) {
      t.cols = (a.cols - c0) / 2;
      t.c = a.c + (long)(c0 / 2) * a.sum;
      t.up = a.up + (long)(c0 / 2) * a.sum;
      t.out = a.out + (long)r0 * (a.cols / 2) + c0 / 2;
    }
    t.part = a.part + (long)u * a.height * gt::TILE;
    if (EXTRA && s == 0) {
      t.r2 = a.r2 + (long)r0 * a.rank;
      t.c2 = a.c2 + (long)c0 * a.rank_c;
      t.rank = a.rank;
      t.rank_c = a.rank_c;
    }
    return t;
  }
};

// SHORT, PARTS, EXTRA, RELU2: gemm_tile.h
template <Form F, bool SHORT, bool PARTS, bool EXTRA = false, bool RELU2 = false>
__global__ __launch_bounds__(gt::THREADS, 1) void linear_tile_kernel(const Args a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  Tiles<F, EXTRA> tiles(a);
  const gt::Shape shape{2u * (F == DW ? a.rows : a.sum), 2u * (F == Y || F == GLU ? a.sum : a.cols),
                        F == GLU ? (unsigned)a.cols : 2u * a.cols};
  gt::Run<F == DW, F == DW || F == DX, Tiles<F, EXTRA>, SHORT, PARTS, EXTRA, RELU2, F == GLU>(tiles, shape, smem)();
}

// us that tiles of `height` rows and sums in `parts` take. A pair of steps of a tile of 32 n rows takes a + b
// n, a little more where all CUs are at work (the card's power); fitted to 114 shapes of either gradient and 5
// heights (1, 2, 3, 4, 6 and 8 parts for two of them): off by 7% (rms), and the choice by it by 0.5% from the
// best one. x w^T: fitted to three or four cuts of 1917 shapes of 100 to 24000 rows; over 3752 others, with all heights and the
// four to six likeliest ways to cut their sums, off by 13%. Where output_own (ops/linear.py) takes the product the choice is off
// by 0.7% in the mean, by 5% and more for one shape in 20, by 22% at most (633 x 14336 -> 3000 78 us, by 256 rows and 6 parts 64).
inline float predicted(Form form, long rows, long cols, long sum, int height, int parts) {
  struct Fit {
    float start, a, b, a_all, b_all, tile, add, add_mb;
  };
  const Fit f = form == DW   ? Fit{5.8f, .104f, .103f, .196f, .141f, 2.36f, 2.6f, .92f}
                : form == DX ? Fit{5.6f, .044f, .109f, .136f, .146f, 1.78f, 4.6f, .88f}
                             : Fit{2.6f, .387f, .0415f, .314f, .1364f, 3.13f, 6.f, .86f};
  const long tiles = (rows + height - 1) / height * ((cols + gt::TILE - 1) / gt::TILE) * parts;
  const float pairs = (sum + 64 * parts - 1) / (64 * parts), n = height / 32;
  const auto round = [&](float busy) {
    return pairs * (f.a + f.b * n + busy * (f.a_all - f.a + (f.b_all - f.b) * n)) + f.tile;
  };
  float t = f.start + tiles / 256 * round(1.f);
  if (tiles % 256) t += round(tiles % 256 / 256.f);
  return parts == 1 ? t : t + f.add + f.add_mb * 1e-6f * rows * cols * parts;
}

// (GLU: sums are whole)
inline void cut(Form form, Args& a) {
  float least = 0.f;
  a.height = 0;
  for (const int parts : {1, 2, 3, 4, 6, 8}) {
    const int per = (a.sum + 64 * parts - 1) / (64 * parts) * 64;
    // each has 4 pairs of steps or more, the last one 2
    if (parts > 1 && (form == GLU || per < 256 || a.sum - (parts - 1) * per < 128)) continue;
    for (int height = 128; height <= gt::TILE; height += 32) {
      const float t = predicted(form, a.rows, a.cols, a.sum, height, parts);
      if (a.height && t >= least) continue;
      least = t;
      a.height = height;
      a.parts = parts;
      a.per = parts == 1 ? a.sum : per;
    }
  }
}

inline long tiles_of(const Args& a) {
  return ((long)(a.rows + a.height - 1) / a.height) * ((a.cols + gt::TILE - 1) / gt::TILE);
}

// linear_dx with an EXTRA product (lora_grad.hip); linear_y, with one or without, and linear_glu (linear_out.hip)
void launch_extra(const Args& a, unsigned blocks, hipStream_t stream);
void launch_out(const Args& a, unsigned blocks, hipStream_t stream);
void launch_glu(const Args& a, unsigned blocks, hipStream_t stream);

}  // namespace lg
}  // namespace amd_ops
