// Which tiles of a grouped product a workgroup of gemm_tile.h computes (gfx950), from the groups' offsets.
//
// A group's rows are cut into equal parts of at most `cap` rows, rounded up to 32: tiles have unequal
// heights, and a few of them make up a workgroup's whole work (128 groups of about 512 rows, 768
// columns: 960 tiles of 6 or 8 times 32 rows for 256 workgroups). Dealt out in their order they take 1.13 to
// 1.7 times as long as they would if all workgroups had as much; the tallest first, each to the workgroup
// with the least so far, 1.02 to 1.1 (routing at random and with unequal experts; the latter worked out on
// the host for the sizes of the layers measured). The groups are so sorted by height, and a wave deals
// all tiles in rounds: a round gives one tile to each workgroup that has least, one XCD's after another's, so that
// tiles of one group, which follow one another, meet in one L2. Every workgroup works all of it out for itself, while
// its first operands come; nothing is shared and nothing has to be cleared.
#pragma once

#include "gemm_tile.h"

namespace amd_ops {

struct GroupedArgs {
  const bf16 *r, *c;                   // operands of the output's rows and columns
  const bf16 *r2, *c2;                 // nn: a second pair, added to the sum
  const bf16* up;                      // GLU: like c
  bf16 *out, *one, *other;             // one, other: GLU's sums
  const int *tile_map, *offs, *n_tiles;
  int n_mtiles, M, N, K, E;            // tile_map's capacity; rows; w is [E, N, K]
  int cap;                             // rows of a tile at most
};

enum Mode { NT, NN, TN, GLU };         // GLU: nt of two weights, silu of the one times the other

constexpr int MAX_GROUPS = 512, MAX_OWN = 513, BINS = 256;

// a minimum over the wave, in every lane
__device__ __forceinline__ int wave_min(int v) {
#define AMD_OPS_MIN_DPP(ctrl, rows) v = min(v, __builtin_amdgcn_update_dpp(v, v, ctrl, rows, 0xf, false))
  AMD_OPS_MIN_DPP(0x111, 0xf);         // row_shr 1, 2, 4, 8: lanes 15, 31, 47, 63 have their 16's
  AMD_OPS_MIN_DPP(0x112, 0xf);
  AMD_OPS_MIN_DPP(0x114, 0xf);
  AMD_OPS_MIN_DPP(0x118, 0xf);
  AMD_OPS_MIN_DPP(0x142, 0xa);         // row_bcast 15, 31
  AMD_OPS_MIN_DPP(0x143, 0xc);
#undef AMD_OPS_MIN_DPP
  return __builtin_amdgcn_readlane(v, 63);
}

// a sum over the lanes up to this one
__device__ __forceinline__ int wave_scan(int v) {
#define AMD_OPS_ADD_DPP(ctrl, rows) v += __builtin_amdgcn_update_dpp(0, v, ctrl, rows, 0xf, false)
  AMD_OPS_ADD_DPP(0x111, 0xf);
  AMD_OPS_ADD_DPP(0x112, 0xf);
  AMD_OPS_ADD_DPP(0x114, 0xf);
  AMD_OPS_ADD_DPP(0x118, 0xf);
  AMD_OPS_ADD_DPP(0x142, 0xa);
  AMD_OPS_ADD_DPP(0x143, 0xc);
#undef AMD_OPS_ADD_DPP
  return v;
}

// how many lanes below this one are in the mask
__device__ __forceinline__ int below(unsigned long mask) {
  return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
}

template <Mode MODE>
struct GroupedTiles {
  struct Group {
    int start, e, row, n;              // tiles of rows before it; which it is, its first row and its rows
  };
  struct Shared {
    Group group[MAX_GROUPS];
    int own[MAX_OWN];                  // before: the groups' offsets
    int n_tiles, n_own, most;
  };
  static constexpr int LEVELS = MODE == TN ? 4 : 8;
  static constexpr int SMEM = gt::SMEM + sizeof(Shared);

  const GroupedArgs& a;
  Shared& s;
  const int nc, nr;
  int k = 0, own = 0, bin, bins, total;

  __device__ __forceinline__ GroupedTiles(const GroupedArgs& a_, char* smem)
      : a(a_), s(*reinterpret_cast<Shared*>(smem + gt::SMEM)),
        nc(((MODE == NT ? a.N : MODE == GLU ? 2 * a.N : a.K) + gt::TILE - 1) / gt::TILE), nr((a.N + gt::TILE - 1) / gt::TILE) {}

  __device__ __forceinline__ int parts(int n) const { return MODE == TN ? nr : (n + a.cap - 1) / a.cap; }
  // 1 to LEVELS: how long a group's tiles take. nt, nn: their rows in 32, 4 at least (equal parts rounded up: from
  // 4 parts on all of them are of the cap, below no part is left over). tn: by the sum, of the largest group's
  __device__ __forceinline__ int level(int n, int most) const {
    if constexpr (MODE == TN) {
      int l = 1;
#pragma unroll
      for (int q = 1; q < LEVELS; ++q) l += n * LEVELS > most * q;
      return l;
    } else {
      const int p32 = 32 * max(parts(n), 1);
      int l = 4;
#pragma unroll
      for (int q = 4; q < LEVELS; ++q) l += n > q * p32;
      return l;
    }
  }
  // in quarters of a step's MFMAs of 32 rows: 128 cycles; a tile has some 6000 besides
  __device__ __forceinline__ int cost(int level, int most) const {
    if constexpr (MODE == TN) return (max(most, 64) + 31) / 32 * 8 / LEVELS * level + 48;
    else return ((MODE == NT || MODE == GLU ? a.K : a.N) + 31) / 32 * (a.r2 ? 2 : 1) * level + 48;
  }

  // sorts the groups, and the first tile
  __device__ __forceinline__ int first() {
    const int lane = threadIdx.x & 63;
    const int* offs = s.own;
    for (int e = threadIdx.x; e <= a.E; e += gt::THREADS) s.own[e] = a.offs[e];
    __syncthreads();
    if (threadIdx.x < 64) {
      int most = 0;
      if (MODE == TN) {
        for (int e = lane; e < a.E; e += 64) most = max(most, offs[e + 1] - offs[e]);
        most = -wave_min(-most);
      }
      int at[LEVELS + 1] = {};         // where the next group of a level goes
      for (int e0 = 0; e0 < a.E; e0 += 64) {
        const int e = e0 + lane, n = e < a.E ? offs[e + 1] - offs[e] : 0, l = e < a.E ? level(n, most) : 0;
#pragma unroll
        for (int q = 1; q < LEVELS; ++q) at[q] += __builtin_popcountl(__ballot(l > q));    // those above
      }
      for (int e0 = 0; e0 < a.E; e0 += 64) {
        const int e = e0 + lane, o = e < a.E ? offs[e] : 0, n = e < a.E ? offs[e + 1] - o : 0;
        const int l = e < a.E ? level(n, most) : 0;
#pragma unroll
        for (int q = 1; q <= LEVELS; ++q) {
          const unsigned long mask = __ballot(l == q);
          if (l == q) s.group[at[q] + below(mask)] = Group{0, e, o, n};
          at[q] += __builtin_popcountl(mask);
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      int before = 0;
      for (int i0 = 0; i0 < a.E; i0 += 64) {
        const int i = i0 + lane, mine = i < a.E ? parts(s.group[i].n) : 0;
        const int sum = wave_scan(mine);
        if (i < a.E) s.group[i].start = before + sum - mine;
        before += __builtin_amdgcn_readlane(sum, 63);
      }
      if (lane == 0) {
        s.n_tiles = before;
        s.most = most;
      }
    }
    __syncthreads();
    total = __builtin_amdgcn_readfirstlane(s.n_tiles) * nc;
    const int per = min((total + 7) / 8, (int)gridDim.x >> 3), x = blockIdx.x & 7, slot = blockIdx.x >> 3;
    bins = per * 8;
    bin = slot < per ? x * per + slot : -1;
    return bin < total ? bin : -1;
  }

  // deals the tiles out
  __device__ __forceinline__ void loaded() {
    const int lane = threadIdx.x & 63;
    if (total <= bins || total > 48 * bins) {          // none more, or so many that any order will do
      own = total <= bins ? 1 : (total - bin + bins - 1) / bins;
      k = total <= bins ? 1 : -1;
      return;
    }
    if (threadIdx.x < 64) {
      const int most = __builtin_amdgcn_readfirstlane(s.most);
      const int mine = lane == bin / (BINS / 64) ? bin % (BINS / 64) : -1;     // where the lane has this workgroup
      int load[BINS / 64], n_own = 0;
#pragma unroll
      for (int j = 0; j < BINS / 64; ++j) load[j] = lane * (BINS / 64) + j < bins ? 0 : 1 << 30;
      int pos = 0;
      while (pos < total) {
        // the groups of one level, from pos on
        const int g = group_of(pos / nc), lv = level(__builtin_amdgcn_readfirstlane(s.group[g].n), most);
        int end = total;
        for (int i0 = 0; i0 < a.E; i0 += 64) {
          const int i = i0 + lane;
          const unsigned long less = __ballot(i > g && i < a.E && level(s.group[i].n, most) < lv);
          if (less) {
            end = __builtin_amdgcn_readfirstlane(s.group[i0 + __builtin_ctzl(less)].start) * nc;
            break;
          }
        }
        const int c = cost(lv, most);
        while (pos < end) {
          int v = load[0];
#pragma unroll
          for (int j = 1; j < BINS / 64; ++j) v = min(v, load[j]);
          const int least = wave_min(v);
          int rank = 0, all = 0;
#pragma unroll
          for (int j = 0; j < BINS / 64; ++j) {
            const unsigned long mask = __ballot(load[j] == least);
            rank += below(mask);
            all += __builtin_popcountl(mask);
          }
          const int left = end - pos;
#pragma unroll
          for (int j = 0; j < BINS / 64; ++j) {
            const bool has = load[j] == least, takes = has && rank < left;
            if (takes && j == mine) s.own[n_own++] = pos + rank;
            load[j] += takes ? c : 0;
            rank += has;
          }
          pos = min(pos + all, end);
        }
      }
      if (mine >= 0) s.n_own = n_own;
    }
    __syncthreads();
    own = __builtin_amdgcn_readfirstlane(s.n_own);
    k = 1;
  }

  __device__ __forceinline__ int next() {
    if (k < 0) {                       // by turns
      bin += bins;
      return bin < total ? bin : -1;
    }
    return k < own ? __builtin_amdgcn_readfirstlane(s.own[k++]) : -1;
  }

  // the group that has tile j of rows: the last one that starts there or before
  __device__ __forceinline__ int group_of(int j) const {
    const int lane = threadIdx.x & 63;
    int n = 0;
    for (int i0 = 0; i0 < a.E; i0 += 64)
      n += __builtin_popcountl(__ballot(i0 + lane < a.E && s.group[i0 + lane].start <= j));
    return n - 1;
  }

  __device__ __forceinline__ gt::Tile get(int id) const {
    int c0 = id % nc * gt::TILE;
    const int j = id / nc, i = MODE == TN ? j / nr : group_of(j);
    const int e = __builtin_amdgcn_readfirstlane(s.group[i].e), row = __builtin_amdgcn_readfirstlane(s.group[i].row);
    const int n = __builtin_amdgcn_readfirstlane(s.group[i].n);
    const int at = j - __builtin_amdgcn_readfirstlane(s.group[i].start);
    gt::Tile t;
    if constexpr (MODE == TN) {
      const int r0 = at * gt::TILE;
      t.rows = a.N - r0;
      t.cols = a.K - c0;
      t.sum = n;
      t.r = a.r + (long)row * a.N + r0;
      t.c = a.c + (long)row * a.K + c0;
      t.out = a.out + ((long)e * a.N + r0) * a.K + c0;
    } else {
      constexpr bool ROWS = MODE == NT || MODE == GLU;
      const int h = 32 * level(n, 0), r0 = row + at * h, sum = ROWS ? a.K : a.N, cols = ROWS ? a.N : a.K;
      if (MODE == GLU) c0 /= 2;
      const long w = (long)e * a.N * a.K + (ROWS ? (long)c0 * a.K : c0);
      t.rows = min(n - at * h, h);
      t.cols = cols - c0;
      t.sum = sum;
      t.r = a.r + (long)r0 * sum;
      t.c = a.c + w;
      if (MODE == NN && a.r2) {
        t.r2 = a.r2 + (long)r0 * sum;
        t.c2 = a.c2 + w;
      }
      t.out = a.out + (long)r0 * cols + c0;
      if (MODE == GLU) {
        t.up = a.up + w;
        t.one = a.one + (long)r0 * cols + c0;
        t.other = a.other + (long)r0 * cols + c0;
      }
    }
    return t;
  }
};

}  // namespace amd_ops
