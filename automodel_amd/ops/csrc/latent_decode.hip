// Latent attention, decode side: a few query rows against the latent cache,
// with the key and value up-projections absorbed into query and output so that
// only the cache row (latent + shared rotated key) is ever read per key.
//
//   latent_decode_prep     q'[r,h] = [ W_uk[h]^T q_unrot | rotated q ], and the
//                          new token's cache row, in one launch
//   latent_decode_attn     split-KV attention of all heads over the cache:
//                          the heads are the columns of 16x16x32 MFMAs, 16 or 32
//                          of them on one staged key tile
//   latent_decode_combine  merges the splits, then applies W_uv per head
//
// Lengths and slots are device tensors: a captured step replays for every
// position. Keys are split evenly over the row's own length.

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include "common.h"
#include "latent_attn.h"
#include "lds_load.h"
#include "ops_api.h"

namespace amd_ops {

void latent_check_rope(const at::Tensor& cos, const at::Tensor& sin, int64_t rot);
void latent_check_cache(const at::Tensor& cache, at::ScalarType dt, int64_t rank, int64_t rot);

typedef __bf16 lat_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 lat_bf16x4 __attribute__((ext_vector_type(4)));
typedef float lat_f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned lat_u32x4 __attribute__((ext_vector_type(4)));    // 16 bytes in flight

// hardware-transposed read: 16 lanes fetch a [4 keys][16 columns] block, lane g
// receives column g (each lane supplies the address of its own 8 bytes)
__device__ __forceinline__ lat_bf16x4 lds_tr16(const char* p) {
  typedef __attribute__((address_space(3))) lat_bf16x4* lds_ptr;
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
      (lds_ptr)(__attribute__((address_space(3))) char*)const_cast<char*>(p));
}

// ---------------------------------------------------------------------------
// prep: blockIdx.x < H * NC absorbs 8*V latent columns of one head for RT rows
// (8 column groups x 32 slices of the head dim, then a reduction); RT more
// workgroups each write a row's latent into the cache. All of it is latency:
// 64 columns per workgroup, so that 32 heads give one to each CU, and no loop
// over rows where a row ends in a barrier (8 rows, 32 heads, rank 512: 13.5 us
// with one workgroup for all rows' latents, 11.3 now).
// ---------------------------------------------------------------------------
constexpr int LP_VECS = 8;
template <typename T, int V, int RT>
__global__ __launch_bounds__(256) void latent_decode_prep_kernel(
    const T* __restrict__ qkv, const T* __restrict__ w_uk, const T* __restrict__ w_norm, float eps,
    const float* __restrict__ cosb, const float* __restrict__ sinb, int n_pos, int cs_stride,
    const int* __restrict__ pos, const int* __restrict__ slot, T* __restrict__ cache, int n_slots,
    int max_len, T* __restrict__ q_out, int R, int H, int dn, int dr, int rank, int NC) {
  extern __shared__ float sm[];
  constexpr int COLS = LP_VECS * V, SLICES = 256 / LP_VECS;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int r0 = blockIdx.y * RT;
  const int hd = dn + dr, RP = pad32(rank), C = RP + pad32(dr);
  const long N = (long)H * hd + rank + dr;
  if ((int)blockIdx.x >= H * NC) {
    const int r = r0 + blockIdx.x - H * NC;
    if (r >= R) return;
    const int p = min(max(pos[r], 0), n_pos - 1);
    const long cr = cache_row(slot[r], pos[r], n_slots, max_len);
    latent_token<T>(qkv + r * N + (long)H * hd, w_norm, eps, cosb + (long)p * cs_stride,
                    sinb + (long)p * cs_stride, rank, dr, cr >= 0 ? cache + cr * C : nullptr,
                    (T*)nullptr, (T*)nullptr, sm);
    return;
  }
  const int h = blockIdx.x / NC, nc = blockIdx.x % NC;
  float* qs = sm;                                 // [RT][dn]
  float* part = sm + RT * dn;                     // [4 waves][RT][COLS]
#pragma unroll
  for (int rr = wid; rr < RT; rr += 4)
    for (int i = lane; i < dn; i += 64)
      qs[rr * dn + i] = r0 + rr < R ? lat_f(qkv[(r0 + rr) * N + h * hd + i]) : 0.f;
  if (nc == 0) {                                  // rotated part and zero padding
    const int half = dr / 2;
#pragma unroll
    for (int rr = wid; rr < RT; rr += 4) {
      const int r = r0 + rr;
      if (r >= R) break;
      T* o = q_out + ((long)r * H + h) * C;
      const T* src = qkv + r * N + h * hd + dn;
      const int p = min(max(pos[r], 0), n_pos - 1);
      for (int i = lane; i < half; i += 64) {
        const float c = cosb[(long)p * cs_stride + i], s = sinb[(long)p * cs_stride + i];
        const float u = lat_f(src[i]), v = lat_f(src[half + i]);
        o[RP + i] = lat_t<T>(u * c - v * s);
        o[RP + half + i] = lat_t<T>(v * c + u * s);
      }
      for (int i = rank + lane; i < RP; i += 64) o[i] = lat_t<T>(0.f);
      for (int i = RP + dr + lane; i < C; i += 64) o[i] = lat_t<T>(0.f);
    }
  }
  __syncthreads();
  const int vec = tid % LP_VECS, slice = tid / LP_VECS;
  const int col = nc * COLS + vec * V;
  float acc[RT][V];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int j = 0; j < V; ++j) acc[r][j] = 0.f;
  if (col < rank) {                               // V divides rank
    const T* wp = w_uk + (long)h * dn * rank + col;
#pragma unroll 4
    for (int d = slice; d < dn; d += SLICES) {
      const LatPack<T, V> w = *reinterpret_cast<const LatPack<T, V>*>(wp + (long)d * rank);
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        const float qv = qs[r * dn + d];
#pragma unroll
        for (int j = 0; j < V; ++j) acc[r][j] = fmaf(qv, lat_f(w.v[j]), acc[r][j]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int j = 0; j < V; ++j) {
      float a = acc[r][j];
#pragma unroll
      for (int d = LP_VECS; d < 64; d *= 2) a += __shfl_xor(a, d);
      if (lane < LP_VECS) part[(wid * RT + r) * COLS + vec * V + j] = a;
    }
  __syncthreads();
  for (int i = tid; i < RT * COLS; i += 256) {
    const int r = r0 + i / COLS, c = nc * COLS + i % COLS;
    if (r >= R || c >= rank) continue;
    float a = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) a += part[w * RT * COLS + i];
    q_out[((long)r * H + h) * C + c] = lat_t<T>(a);
  }
}

// The same on the matrix cores, for bf16, a head dim in steps of 32 and rows in
// whole 16-byte pieces: 16 rows at once, 64 columns of one head per workgroup, 16
// per wave; W_uk goes through LDS to be read transposed. With rows in registers the
// instructions themselves, each run once, took most of the time: 11.3 us for 8 rows,
// 32 heads, 4.7 here; 1 row, 16 heads 3.6 and 3.4.
constexpr int LPM_STRIDE = 64 * 2 + 16;           // LDS bytes per row of W_uk
__global__ __launch_bounds__(256) void latent_decode_prep_mfma_kernel(
    const bf16* __restrict__ qkv, const bf16* __restrict__ w_uk, const bf16* __restrict__ w_norm,
    float eps, const float* __restrict__ cosb, const float* __restrict__ sinb, int n_pos,
    int cs_stride, const int* __restrict__ pos, const int* __restrict__ slot,
    bf16* __restrict__ cache, int n_slots, int max_len, bf16* __restrict__ q_out, int R, int H,
    int dn, int dr, int rank, int NC) {
  extern __shared__ __attribute__((aligned(16))) char lds[];    // [dn][LPM_STRIDE]
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int lo16 = lane & 15, hi4 = lane >> 4;
  const int r0 = blockIdx.y * 16;
  const int hd = dn + dr, RP = pad32(rank), C = RP + pad32(dr);
  const long N = (long)H * hd + rank + dr;
  if ((int)blockIdx.x >= H * NC) {                // a row's latent
    const int r = r0 + blockIdx.x - H * NC;
    if (r >= R) return;
    const int p = min(max(pos[r], 0), n_pos - 1);
    const long cr = cache_row(slot[r], pos[r], n_slots, max_len);
    latent_token<bf16>(qkv + r * N + (long)H * hd, w_norm, eps, cosb + (long)p * cs_stride,
                       sinb + (long)p * cs_stride, rank, dr, cr >= 0 ? cache + cr * C : nullptr,
                       (bf16*)nullptr, (bf16*)nullptr, reinterpret_cast<float*>(lds));
    return;
  }
  const int h = blockIdx.x / NC, nc = blockIdx.x % NC;
  const bf16* wp = w_uk + (long)h * dn * rank;
#pragma unroll 4
  for (int i = tid; i < dn * 8; i += 256) {
    const int d = i >> 3, col = nc * 64 + (i & 7) * 8;
    lat_u32x4 x = {0u, 0u, 0u, 0u};
    if (col < rank) x = *reinterpret_cast<const lat_u32x4*>(wp + (long)d * rank + col);
    *reinterpret_cast<lat_u32x4*>(lds + d * LPM_STRIDE + (i & 7) * 16) = x;
  }
  // the head's NC workgroups share the rows' rotated part and zero padding
  for (int rr = nc * 4 + wid; rr < 16 && r0 + rr < R; rr += 4 * NC) {
    const int r = r0 + rr, half = dr / 2;
    bf16* o = q_out + ((long)r * H + h) * C;
    const bf16* src = qkv + r * N + h * hd + dn;
    const int p = min(max(pos[r], 0), n_pos - 1);
    for (int i = lane; i < half; i += 64) {
      const float c = cosb[(long)p * cs_stride + i], s = sinb[(long)p * cs_stride + i];
      const float u = bf2f(src[i]), v = bf2f(src[half + i]);
      o[RP + i] = f2bf(u * c - v * s);
      o[RP + half + i] = f2bf(v * c + u * s);
    }
    for (int i = rank + lane; i < RP; i += 64) o[i] = f2bf(0.f);
    for (int i = RP + dr + lane; i < C; i += 64) o[i] = f2bf(0.f);
  }
  __syncthreads();
  const int r = r0 + lo16;
  const bf16* qp = qkv + min(r, R - 1) * N + h * hd + hi4 * 8;
  const char* wl = lds + (hi4 * 8 + (lo16 >> 2)) * LPM_STRIDE + wid * 32 + (lo16 & 3) * 8;
  lat_f32x4 acc = {0.f, 0.f, 0.f, 0.f};           // D[column = 4 hi4 + i][row = lo16]
#pragma unroll 4
  for (int d = 0; d < dn; d += 32) {
    const lat_bf16x8 qv = __builtin_bit_cast(lat_bf16x8, *reinterpret_cast<const lat_u32x4*>(qp + d));
    const lat_bf16x4 w0 = lds_tr16(wl + d * LPM_STRIDE), w1 = lds_tr16(wl + (d + 4) * LPM_STRIDE);
    const lat_bf16x8 wv = __builtin_shufflevector(w0, w1, 0, 1, 2, 3, 4, 5, 6, 7);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, qv, acc, 0, 0, 0);
  }
  const int col = nc * 64 + wid * 16 + hi4 * 4;
  if (r < R && col < rank) {                      // rank % 8 == 0: all 4 columns or none
    bf16x4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) y.v[i] = f2bf(acc[i]);
    *reinterpret_cast<bf16x4*>(q_out + ((long)r * H + h) * C + col) = y;
  }
}

// ---------------------------------------------------------------------------
// attention over the cache. grid (splits, head groups of 16 HT, rows)
// ---------------------------------------------------------------------------
constexpr int LD_KEYS = 64;           // keys per tile: 4 waves x 16
constexpr int LD_PSTRIDE = LD_KEYS * 2 + 16;

// HT: head tiles of 16 per workgroup, four waves each; they share the staged keys.
// NCT: 16-column value tiles per wave (4 waves cover RP <= 64 * NCT). NPM: bound on
// the 32-column steps of a row. One head tile has one tile of keys in LDS, which
// leaves room for a second workgroup; two have a second buffer, whose loads are in
// flight while the first one is used.
//
// With few rows a split is a tile or two, so this is a chain of latencies, and of
// instructions that run once: both products put the head in the lane (columns of the
// accumulator), so that the running maximum and scale are one value a lane, P goes
// to LDS in one piece and the partial results leave in 16-byte stores; keys go to
// LDS without registers in between; the queries sit in registers, which leaves LDS
// for two workgroups per CU. With heads in the accumulator's rows, keys through
// registers and queries in LDS: 9.5 us for 1 row, 16 heads, 200 keys and 21.0 for 8
// rows, 32 heads, 1500 keys; now 7.2 and 12.3. (Rows of 576 columns, 512 of them
// latents. 32 rows of 32000 keys, 32 heads, read at the memory's rate: 300 with the
// launches around it, now 307.)
template <int NCT, int NPM, int HT>
__global__ __launch_bounds__(256 * HT) void latent_decode_attn_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ cache, const int* __restrict__ slot,
    const int* __restrict__ pos, float* __restrict__ part_o, float* __restrict__ part_ml,
    int n_slots, int max_len, int H, int RP, int C, float scale) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int KS = C * 2;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wid = wave & 3, ht = wave >> 2;       // part of the keys and columns; head tile
  const int tile_bytes = LD_KEYS * KS;
  char* kt = lds;                                 // [64][KS], HT times
  const unsigned kt_at = fa::lds_address(lds);
  char* pt = lds + HT * tile_bytes + ht * 16 * (LD_PSTRIDE + 16);   // [16][LD_PSTRIDE]
  float* red = reinterpret_cast<float*>(pt + 16 * LD_PSTRIDE);      // [4][16]
  const int lo16 = lane & 15, hi4 = lane >> 4;
  const int split = blockIdx.x, n_split = gridDim.x;
  const int h = (blockIdx.y * HT + ht) * 16 + lo16;   // this lane's head
  const int r = blockIdx.z;

  const int steps = C / 32;
  lat_bf16x8 qf[NPM];                             // step j: columns 32j + 8 hi4 of head h
  {
    const bf16* qp = q + ((long)r * H + min(h, H - 1)) * C + hi4 * 8;
#pragma unroll
    for (int j = 0; j < NPM; ++j)
      if (j < steps)                              // uniform
        qf[j] = __builtin_bit_cast(lat_bf16x8, *reinterpret_cast<const lat_u32x4*>(qp + j * 32));
  }

  const int sl = slot[r];
  const int n = (sl < 0 || sl >= n_slots) ? 0 : min(max(pos[r] + 1, 0), max_len);
  const int tiles = (n + LD_KEYS - 1) / LD_KEYS;
  const int per = (tiles + n_split - 1) / n_split;
  const int t_lo = split * per, t_hi = min(t_lo + per, tiles);
  const bf16* base = cache + (long)(n > 0 ? sl : 0) * max_len * C;

  // A tile lies in LDS without padding, row after row; piece c of row r sits at
  // c ^ swz(r), which spreads the 16 rows of a read over the banks: the rows'
  // starts repeat every 16 / g rows, g pieces apart (g: the largest power of two in
  // a row's pieces, 16 at most)
  const int vecs = C / 8;                         // 16-byte pieces per row, a multiple of 4
  const int lg = min(__builtin_ctz(vecs), 4), sh = 4 - lg, gm = (1 << lg) - 1;
  const unsigned magic = ((1u << 20) + vecs - 1) / vecs;    // i / vecs, exact for i < 128 vecs
  auto stage = [&](int t, int buf) {
    const bf16* tile = base + (long)t * LD_KEYS * C;
    const int left = n - t * LD_KEYS;             // rows past the end: masked below
#pragma unroll 2
    for (int j = wave; j < vecs; j += 4 * HT) {   // a kilobyte each
      const unsigned i = j * 64 + lane, row = (i * magic) >> 20, c = i - row * vecs;
      const unsigned off = (unsigned)min((int)row, left - 1) * C * 2 + ((c ^ ((row >> sh) & gm)) << 4);
      fa::load_lds16(kt_at + buf * tile_bytes + j * 1024, tile, off);
    }
  };
  // pieces of this lane's reads: row lo16 of a wave's keys; rows hi4 * 8 + lo16 / 4 and 4 on
  const int ks_swz = (lo16 >> sh) & gm;
  const int v_row = (hi4 & 1) * 8 + (lo16 >> 2), v_swz0 = (v_row >> sh) & gm,
            v_swz1 = ((v_row + 4) >> sh) & gm;

  lat_f32x4 acc[NCT];
  float m_run = -1e30f, l_run = 0.f;
#pragma unroll
  for (int c = 0; c < NCT; ++c) acc[c] = lat_f32x4{0.f, 0.f, 0.f, 0.f};

  if (HT == 2 && t_lo < t_hi) stage(t_lo, 0);
  for (int t = t_lo; t < t_hi; ++t) {
    const int k0 = t * LD_KEYS;
    if (HT == 2) kt = lds + ((t - t_lo) & 1) * tile_bytes;
    else stage(t, 0);

    fa::wait_loads();
    fa::barrier();
    if (HT == 2 && t + 1 < t_hi) stage(t + 1, (t + 1 - t_lo) & 1);

    // scores: D[key = 4 hi4 + i][head = lo16] of this wave's 16 keys
    lat_f32x4 s = {0.f, 0.f, 0.f, 0.f};
    const char* kp = kt + (wid * 16 + lo16) * KS;
#pragma unroll
    for (int j = 0; j < NPM; ++j)
      if (j < steps) {
        const lat_bf16x8 k =
            *reinterpret_cast<const lat_bf16x8*>(kp + (((j * 4 + hi4) ^ ks_swz) << 4));
        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, qf[j], s, 0, 0, 0);
      }
    float mx = -1e30f;
    bool live[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      live[i] = k0 + wid * 16 + hi4 * 4 + i < n;
      s[i] = live[i] ? s[i] * scale : -1e30f;
      mx = fmaxf(mx, s[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    if (hi4 == 0) red[wid * 16 + lo16] = mx;
    fa::barrier();
    float mn = m_run;
#pragma unroll
    for (int w = 0; w < 4; ++w) mn = fmaxf(mn, red[w * 16 + lo16]);
    const float alpha = __expf(m_run - mn);
    m_run = mn;
    bf16x4 p;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float e = live[i] ? __expf(s[i] - mn) : 0.f;
      sum += e;
      p.v[i] = f2bf(e);
    }
    l_run = l_run * alpha + sum;
    *reinterpret_cast<bf16x4*>(pt + lo16 * LD_PSTRIDE + (wid * 16 + hi4 * 4) * 2) = p;
#pragma unroll
    for (int c = 0; c < NCT; ++c) acc[c] *= alpha;
    fa::barrier();

    // O[column][head] += V[key][column] P[head][key], V = the tile's latents
#pragma unroll 1
    for (int ks = 0; ks < LD_KEYS / 32; ++ks) {
      const lat_bf16x8 p8 = *reinterpret_cast<const lat_bf16x8*>(pt + lo16 * LD_PSTRIDE +
                                                                 (ks * 32 + hi4 * 8) * 2);
#pragma unroll
      for (int c = 0; c < NCT; ++c) {
        const int n0 = (wid * NCT + c) * 16;
        if (n0 < RP) {                            // wave-uniform
          const char* vp = kt + (ks * 32 + hi4 * 8 + (lo16 >> 2)) * KS + (lo16 & 1) * 8;
          const int piece = n0 / 8 + ((lo16 & 3) >> 1);
          const lat_bf16x4 v0 = lds_tr16(vp + ((piece ^ v_swz0) << 4));
          const lat_bf16x4 v1 = lds_tr16(vp + 4 * KS + ((piece ^ v_swz1) << 4));
          const lat_bf16x8 v = __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7);
          acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, p8, acc[c], 0, 0, 0);
        }
      }
    }
    if (HT == 1) fa::barrier();                   // before the tile is overwritten
  }

  // partial results of this split; an empty split stores zeros
  l_run += __shfl_xor(l_run, 16);
  l_run += __shfl_xor(l_run, 32);
  if (hi4 == 0) red[wid * 16 + lo16] = l_run;
  fa::barrier();
  if (h >= H) return;
  const long o = ((long)r * H + h) * n_split + split;
  if (wid == 0 && hi4 == 0) {
    float l = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) l += red[w * 16 + lo16];
    part_ml[o * 2] = m_run;
    part_ml[o * 2 + 1] = l;
  }
#pragma unroll
  for (int c = 0; c < NCT; ++c) {
    const int n0 = (wid * NCT + c) * 16;
    if (n0 < RP) *reinterpret_cast<lat_f32x4*>(part_o + o * RP + n0 + hi4 * 4) = acc[c];
  }
}

// ---------------------------------------------------------------------------
// merge: grid (column chunks of 128, H, R). Splits -> normalised latent output
// in f32; 32 threads cover the columns, 8 groups of them share the splits.
// ---------------------------------------------------------------------------
constexpr int LM_COLS = 128;
__global__ __launch_bounds__(256) void latent_decode_merge_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml, float* __restrict__ o,
    int H, int RP, int S) {
  extern __shared__ float sm[];
  float* wt = sm;                                 // [S]
  lat_f32x4* half = reinterpret_cast<lat_f32x4*>(sm + (S + 3) / 4 * 4);    // [8][32]
  const int tid = threadIdx.x, lane = tid & 63;
  const long rh = (long)blockIdx.z * H + blockIdx.y;
  const float* ml = part_ml + rh * S * 2;
  if (tid < 64) {                                 // one wave weighs the splits
    float m = -1e30f;
    for (int s = lane; s < S; s += 64) m = fmaxf(m, ml[2 * s]);
    m = wave_reduce_max(m);
    float l = 0.f;
    for (int s = lane; s < S; s += 64) l += __expf(ml[2 * s] - m) * ml[2 * s + 1];
    l = wave_reduce_sum(l);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    for (int s = lane; s < S; s += 64) wt[s] = __expf(ml[2 * s] - m) * inv;
  }
  __syncthreads();
  const int col = blockIdx.x * LM_COLS + (tid & 31) * 4, g = tid >> 5;
  lat_f32x4 a = {0.f, 0.f, 0.f, 0.f};
  if (col < RP) {                                 // RP % 32 == 0
    const float* po = part_o + rh * S * RP + col;
#pragma unroll 8
    for (int s = g; s < S; s += 8)
      a += wt[s] * *reinterpret_cast<const lat_f32x4*>(po + (long)s * RP);
  }
  half[g * 32 + (tid & 31)] = a;
  __syncthreads();
  if (g == 0 && col < RP) {
#pragma unroll
    for (int i = 1; i < 8; ++i) a += half[i * 32 + tid];
    *reinterpret_cast<lat_f32x4*>(o + rh * RP + col) = a;
  }
}

// ---------------------------------------------------------------------------
// value up-projection: grid (value chunks of 32, H, row groups of RT). A wave
// takes 8 rows of W_uv[h] at once against the latent outputs in LDS.
// ---------------------------------------------------------------------------
constexpr int LC_ROWS = 32;
template <typename T, int V, int RT>
__global__ __launch_bounds__(256) void latent_decode_value_kernel(
    const float* __restrict__ o_lat, const T* __restrict__ w_uv, T* __restrict__ out, int R, int H,
    int dv, int rank, int stride) {
  extern __shared__ float sm[];                   // [RT][rank]
  constexpr int NV = LC_ROWS / 4;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int h = blockIdx.y, r0 = blockIdx.z * RT;
  const int nc = rank / V;                        // column c = chunk * V + j sits at [j][chunk]
  for (int i = tid; i < RT * rank; i += 256) {
    const int rr = i / rank, c = i % rank, r = min(r0 + rr, R - 1);
    sm[rr * rank + (c % V) * nc + c / V] = o_lat[((long)r * H + h) * stride + c];
  }
  const int v0 = blockIdx.x * LC_ROWS + wid * NV;
  const T* w[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) w[v] = w_uv + ((long)h * dv + min(v0 + v, dv - 1)) * rank;
  float acc[NV * RT];
#pragma unroll
  for (int i = 0; i < NV * RT; ++i) acc[i] = 0.f;
  __syncthreads();
  for (int c = lane; c < nc; c += 64) {
    LatPack<T, V> x[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) x[v] = *reinterpret_cast<const LatPack<T, V>*>(w[v] + c * V);
#pragma unroll
    for (int rr = 0; rr < RT; ++rr)
#pragma unroll
      for (int j = 0; j < V; ++j) {
        const float o = sm[rr * rank + j * nc + c];
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[rr * NV + v] = fmaf(lat_f(x[v].v[j]), o, acc[rr * NV + v]);
      }
  }
  // all NV * RT sums over the wave at once: halve the set at every step, so
  // that lane l ends with sum l / (64 / (NV * RT))
  constexpr int NA = NV * RT;
  int mask = 32;
#pragma unroll
  for (int n = NA; n > 1; n /= 2, mask /= 2) {
    const bool up = lane & mask;
#pragma unroll
    for (int i = 0; i < n / 2; ++i) {
      const float keep = up ? acc[i + n / 2] : acc[i], give = up ? acc[i] : acc[i + n / 2];
      acc[i] = keep + __shfl_xor(give, mask);
    }
  }
  for (; mask > 0; mask /= 2) acc[0] += __shfl_xor(acc[0], mask);
  const int idx = lane / (64 / NA), rr = idx / NV, v = idx % NV;
  if (lane % (64 / NA) == 0 && v0 + v < dv && r0 + rr < R)
    out[((long)(r0 + rr) * H + h) * dv + v0 + v] = lat_t<T>(acc[0]);
}

// The same on the matrix cores, for bf16 weights and a rank in whole 16-byte
// pieces: grid (value chunks of 16, H, row groups of 16), the four waves share
// the rank. The outputs stay float32: as the sum of three bf16 parts, 24 bits,
// they enter the products exactly. 8 rows, 32 heads, 24 splits: 18.9 us with the
// merge above by the kernel above, 8.3 now.
__global__ __launch_bounds__(256) void latent_decode_value_mfma_kernel(
    const float* __restrict__ o_lat, const bf16* __restrict__ w_uv, bf16* __restrict__ out, int R,
    int H, int dv, int rank, int stride) {
  __shared__ float red[4][16][17];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int lo16 = lane & 15, hi4 = lane >> 4;
  const int h = blockIdx.y, v0 = blockIdx.x * 16, r0 = blockIdx.z * 16;
  const float* o = o_lat + ((long)min(r0 + lo16, R - 1) * H + h) * stride;
  const bf16* w = w_uv + ((long)h * dv + min(v0 + lo16, dv - 1)) * rank;
  lat_f32x4 acc = {0.f, 0.f, 0.f, 0.f};           // D[value = 4 hi4 + i][row = lo16]
#pragma unroll 2
  for (int k0 = wid * 32; k0 < rank; k0 += 128) {
    const int k = k0 + hi4 * 8;
    lat_bf16x8 wv = {}, part[3] = {};
    if (k < rank) {                               // all 8 columns or none
      wv = __builtin_bit_cast(lat_bf16x8, *reinterpret_cast<const lat_u32x4*>(w + k));
      const lat_f32x4 x[2] = {*reinterpret_cast<const lat_f32x4*>(o + k),
                              *reinterpret_cast<const lat_f32x4*>(o + k + 4)};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float f = x[j / 4][j % 4];
        part[0][j] = (__bf16)f;
        // nothing is left of an infinity
        const float mid = __builtin_isfinite(f) ? f - (float)part[0][j] : 0.f;
        part[1][j] = (__bf16)mid;
        part[2][j] = (__bf16)(mid - (float)part[1][j]);
      }
    }
#pragma unroll
    for (int i = 2; i >= 0; --i)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, part[i], acc, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) red[wid][lo16][hi4 * 4 + i] = acc[i];
  __syncthreads();
  const int r = tid >> 4, v = tid & 15;
  if (r0 + r < R && v0 + v < dv)
    out[((long)(r0 + r) * H + h) * dv + v0 + v] =
        f2bf(red[0][r][v] + red[1][r][v] + red[2][r][v] + red[3][r][v]);
}

// Few rows and splits: merge and up-projection in one launch, grid (value chunks of
// 16, H, R). A lane adds up the splits of its own columns, which no other lane of
// the wave needs, and every workgroup does so again. 1 row, 16 heads, 4 splits: 7.6 us
// in two launches, 4.1 now; 24 splits, 32 heads 8.2, and 7.4 by the kernels above.
__global__ __launch_bounds__(256) void latent_decode_value_fold_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml,
    const bf16* __restrict__ w_uv, bf16* __restrict__ out, int H, int dv, int rank, int stride,
    int S) {
  constexpr int V = 8, NV = 4;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int h = blockIdx.y, v0 = blockIdx.x * 16 + wid * NV;
  const long rh = (long)blockIdx.z * H + h;
  const float* ml = part_ml + rh * S * 2;
  const bf16* w[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) w[v] = w_uv + ((long)h * dv + min(v0 + v, dv - 1)) * rank;
  float acc[NV] = {};
  float m = -1e30f, l = 0.f;
  for (int s = 0; s < S; ++s) m = fmaxf(m, ml[2 * s]);
  for (int s = 0; s < S; ++s) l = fmaf(__expf(ml[2 * s] - m), ml[2 * s + 1], l);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  for (int c = lane * V; c < rank; c += 64 * V) {           // V divides rank
    LatPack<bf16, V> x[NV];
    LatPack<float, V> o = {};
#pragma unroll
    for (int v = 0; v < NV; ++v) x[v] = *reinterpret_cast<const LatPack<bf16, V>*>(w[v] + c);
#pragma unroll 4
    for (int s = 0; s < S; ++s) {
      const float e = __expf(ml[2 * s] - m) * inv;
      const LatPack<float, V> po =
          *reinterpret_cast<const LatPack<float, V>*>(part_o + (rh * S + s) * stride + c);
#pragma unroll
      for (int j = 0; j < V; ++j) o.v[j] = fmaf(e, po.v[j], o.v[j]);
    }
#pragma unroll
    for (int j = 0; j < V; ++j)
#pragma unroll
      for (int v = 0; v < NV; ++v) acc[v] = fmaf(bf2f(x[v].v[j]), o.v[j], acc[v]);
  }
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const float t = wave_reduce_sum(acc[v]);
    if (lane == 0 && v0 + v < dv) out[rh * dv + v0 + v] = f2bf(t);
  }
}

// ---------------------------------------------------------------------------
namespace {
bool dec_t(const at::Tensor& x) {
  return x.is_cuda() && x.is_contiguous() &&
         (x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kFloat);
}
bool dec_i32(const at::Tensor& x, int64_t n) {
  return x.is_cuda() && x.is_contiguous() && x.scalar_type() == at::kInt && x.numel() == n;
}
constexpr size_t LDS_MAX = 160 * 1024;
bool aligned(const at::Tensor& x) { return reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0; }
}  // namespace

#define ROW_TILE(R, ...)                                   \
  do {                                                     \
    if ((R) <= 1) { constexpr int RT = 1; __VA_ARGS__ }           \
    else if ((R) <= 2) { constexpr int RT = 2; __VA_ARGS__ }      \
    else if ((R) <= 4) { constexpr int RT = 4; __VA_ARGS__ }      \
    else { constexpr int RT = 8; __VA_ARGS__ }                    \
  } while (0)

at::Tensor latent_decode_prep(const at::Tensor& qkv, const at::Tensor& w_uk,
                              const at::Tensor& w_norm, double eps, const at::Tensor& cos,
                              const at::Tensor& sin, const at::Tensor& pos, const at::Tensor& slot,
                              at::Tensor cache, int64_t heads, int64_t dn, int64_t dr) {
  TORCH_CHECK(dec_t(qkv) && qkv.dim() == 2, "latent_decode_prep: qkv [R, N]");
  const auto dt = qkv.scalar_type();
  const int64_t R = qkv.size(0), rank = w_norm.numel();
  TORCH_CHECK(dec_t(w_uk) && w_uk.scalar_type() == dt && w_uk.dim() == 2 &&
                  w_uk.size(0) == heads * dn && w_uk.size(1) == rank,
              "latent_decode_prep: W_uk [heads * dim, rank]");
  TORCH_CHECK(dec_t(w_norm) && w_norm.scalar_type() == dt, "latent_decode_prep: norm weight");
  TORCH_CHECK(qkv.size(1) == heads * (dn + dr) + rank + dr, "latent_decode_prep: qkv width");
  TORCH_CHECK(dec_i32(pos, R) && dec_i32(slot, R), "latent_decode_prep: pos/slot int32 [R]");
  latent_check_rope(cos, sin, dr);
  latent_check_cache(cache, dt, rank, dr);
  auto q = at::empty({R, heads, cache.size(2)}, qkv.options());
  if (R == 0) return q;
  auto stream = c10::hip::getCurrentHIPStream();
  const bool vec = rank % 8 == 0;
  if (dt == at::kBFloat16 && vec && dn % 32 == 0 && dn <= 256 && (dn + dr) % 8 == 0 &&
      qkv.size(1) % 8 == 0 && aligned(qkv) && aligned(w_uk)) {
    const int NC = (int)((rank + 63) / 64);
    latent_decode_prep_mfma_kernel<<<dim3(heads * NC + std::min<int64_t>(R, 16), (R + 15) / 16),
                                     dim3(256), dn * LPM_STRIDE, stream>>>(
        reinterpret_cast<const bf16*>(qkv.data_ptr()), reinterpret_cast<const bf16*>(w_uk.data_ptr()),
        reinterpret_cast<const bf16*>(w_norm.data_ptr()), (float)eps, cos.data_ptr<float>(),
        sin.data_ptr<float>(), (int)cos.size(0), (int)cos.size(1), pos.data_ptr<int>(),
        slot.data_ptr<int>(), reinterpret_cast<bf16*>(cache.data_ptr()), (int)cache.size(0),
        (int)cache.size(1), reinterpret_cast<bf16*>(q.data_ptr()), (int)R, (int)heads, (int)dn,
        (int)dr, (int)rank, NC);
    HIP_CHECK_KERNEL();
    return q;
  }
  const int cols = LP_VECS * (vec ? 8 : 1);
  const int NC = (int)((rank + cols - 1) / cols);
#define LAUNCH(TT, VV)                                                                           \
  latent_decode_prep_kernel<TT, VV, RT>                                                          \
      <<<dim3(heads * NC + RT, (R + RT - 1) / RT), dim3(256), smem, stream>>>(                   \
          reinterpret_cast<const TT*>(qkv.data_ptr()),                                           \
          reinterpret_cast<const TT*>(w_uk.data_ptr()),                                          \
          reinterpret_cast<const TT*>(w_norm.data_ptr()), (float)eps, cos.data_ptr<float>(),     \
          sin.data_ptr<float>(), (int)cos.size(0), (int)cos.size(1), pos.data_ptr<int>(),        \
          slot.data_ptr<int>(), reinterpret_cast<TT*>(cache.data_ptr()), (int)cache.size(0),     \
          (int)cache.size(1), reinterpret_cast<TT*>(q.data_ptr()), (int)R, (int)heads, (int)dn,  \
          (int)dr, (int)rank, NC)
  ROW_TILE(R, {
    const size_t smem = (RT * dn + 4 * RT * cols + 16) * sizeof(float);
    TORCH_CHECK(smem <= 64 * 1024, "latent_decode_prep: head dim too large");
    if (dt == at::kBFloat16) {
      if (vec) LAUNCH(bf16, 8); else LAUNCH(bf16, 1);
    } else {
      if (vec) LAUNCH(float, 8); else LAUNCH(float, 1);
    }
  });
#undef LAUNCH
  HIP_CHECK_KERNEL();
  return q;
}

// q [R, H, C] from latent_decode_prep -> (part_o [R, H, S, RP], part_ml [R, H, S, 2])
std::tuple<at::Tensor, at::Tensor> latent_decode_attn(const at::Tensor& q, const at::Tensor& cache,
                                                      const at::Tensor& slot, const at::Tensor& pos,
                                                      int64_t rank, int64_t rot, double scale,
                                                      int64_t splits) {
  TORCH_CHECK(dec_t(q) && q.dim() == 3 && q.scalar_type() == at::kBFloat16,
              "latent_decode_attn: q [R,H,C] bf16");
  latent_check_cache(cache, at::kBFloat16, rank, rot);
  const int64_t R = q.size(0), H = q.size(1), C = q.size(2), RP = pad32(rank);
  TORCH_CHECK(C == cache.size(2) && RP <= 512, "latent_decode_attn: rank <= 512");
  TORCH_CHECK(dec_i32(pos, R) && dec_i32(slot, R), "latent_decode_attn: pos/slot int32 [R]");
  TORCH_CHECK(splits >= 1 && splits <= 1024 && R <= 65535, "latent_decode_attn: splits/rows");
  auto part_o = at::empty({R, H, splits, RP}, q.options().dtype(at::kFloat));
  auto part_ml = at::empty({R, H, splits, 2}, part_o.options());
  if (R == 0) return {part_o, part_ml};
  auto stream = c10::hip::getCurrentHIPStream();
  auto smem_of = [&](int ht) { return (size_t)ht * (LD_KEYS * C * 2 + 16 * (LD_PSTRIDE + 16)); };
  TORCH_CHECK(smem_of(1) <= LDS_MAX, "latent_decode_attn: tile exceeds LDS");
  // Pairs of head tiles read every key once for 32 heads and load while they work, but take a
  // whole CU. They win from 64 rows on, where splits are long (one head tile and pairs, prep
  // and combine included: 64 rows of 16000 keys, 32 heads 350 and 313 us, 128 heads 1312 and
  // 1076; of 500 keys 45 and 44, 132 and 125), and lose below (32 rows of 2000 keys, 64 heads
  // 66.8 and 70.3; 1 of 200, 32 heads 15.6 and 18.6), or where their last pass leaves more of the
  // chip idle (96 rows of 8000, 128 heads, 256 latents: 620 and 712; 128 rows: 918 and 741).
  auto fill = [&](int ht) {
    const int64_t round = 256 * (LDS_MAX / smem_of(ht));
    const int64_t n = R * ((H + 16 * ht - 1) / (16 * ht)) * splits;
    return (double)n / ((n + round - 1) / round * round);
  };
  const bool pairs = H > 16 && R >= 64 && smem_of(2) <= LDS_MAX && fill(2) >= fill(1);
  const size_t smem = smem_of(pairs ? 2 : 1);
#define LAUNCH(NCT, NPM, HT)                                                                     \
  do {                                                                                           \
    static const hipError_t attr_ = hipFuncSetAttribute(                                         \
        reinterpret_cast<const void*>(&latent_decode_attn_kernel<NCT, NPM, HT>),                 \
        hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_MAX);                               \
    TORCH_CHECK(attr_ == hipSuccess, "latent_decode_attn: LDS attribute");                       \
    latent_decode_attn_kernel<NCT, NPM, HT>                                                      \
        <<<dim3(splits, (H + 16 * HT - 1) / (16 * HT), R), dim3(256 * HT), smem, stream>>>(      \
            reinterpret_cast<const bf16*>(q.data_ptr()),                                         \
            reinterpret_cast<const bf16*>(cache.data_ptr()), slot.data_ptr<int>(),               \
            pos.data_ptr<int>(), part_o.data_ptr<float>(), part_ml.data_ptr<float>(),            \
            (int)cache.size(0), (int)cache.size(1), (int)H, (int)RP, (int)C, (float)scale);      \
  } while (0)
  TORCH_CHECK(C / 32 <= 26, "latent_decode_attn: latent and rotated key too wide");
  if (RP <= 128 && C <= 256) { if (pairs) LAUNCH(2, 8, 2); else LAUNCH(2, 8, 1); }
  else if (RP <= 256 && C <= 384) { if (pairs) LAUNCH(4, 12, 2); else LAUNCH(4, 12, 1); }
  else if (C <= 640) { if (pairs) LAUNCH(8, 20, 2); else LAUNCH(8, 20, 1); }
  else LAUNCH(8, 26, 1);
#undef LAUNCH
  HIP_CHECK_KERNEL();
  return {part_o, part_ml};
}

// part_o [R, H, S, stride >= rank] f32 (+ part_ml) and W_uv [H * dv, rank] -> [R, H * dv]
at::Tensor latent_decode_combine(const at::Tensor& part_o,
                                 const std::optional<at::Tensor>& part_ml, const at::Tensor& w_uv,
                                 int64_t dv) {
  TORCH_CHECK(part_o.is_cuda() && part_o.is_contiguous() && part_o.dim() == 4 &&
                  part_o.scalar_type() == at::kFloat,
              "latent_decode_combine: part_o [R,H,S,n] f32");
  const int64_t R = part_o.size(0), H = part_o.size(1), S = part_o.size(2), n = part_o.size(3);
  TORCH_CHECK(dec_t(w_uv) && w_uv.dim() == 2 && w_uv.size(0) == H * dv && w_uv.size(1) <= n,
              "latent_decode_combine: W_uv [H * dv, rank]");
  const int64_t rank = w_uv.size(1);
  if (part_ml) {
    TORCH_CHECK(part_ml->is_cuda() && part_ml->is_contiguous() &&
                    part_ml->scalar_type() == at::kFloat && part_ml->numel() == R * H * S * 2,
                "latent_decode_combine: part_ml [R,H,S,2] f32");
  } else {
    TORCH_CHECK(S == 1, "latent_decode_combine: splits need part_ml");
  }
  auto out = at::empty({R, H * dv}, w_uv.options());
  if (R == 0) return out;
  auto stream = c10::hip::getCurrentHIPStream();
  const bool vec = rank % 8 == 0;
  const bool wide = vec && w_uv.scalar_type() == at::kBFloat16 && n % 4 == 0 && aligned(part_o) &&
                    aligned(w_uv);
  TORCH_CHECK(!part_ml || (n % 32 == 0 && S <= 1024),
              "latent_decode_combine: padded rank, splits <= 1024");
  if (wide && part_ml && R * S <= 20) {
    latent_decode_value_fold_kernel<<<dim3((dv + 15) / 16, H, R), dim3(256), 0, stream>>>(
        part_o.data_ptr<float>(), part_ml->data_ptr<float>(),
        reinterpret_cast<const bf16*>(w_uv.data_ptr()), reinterpret_cast<bf16*>(out.data_ptr()),
        (int)H, (int)dv, (int)rank, (int)n, (int)S);
    HIP_CHECK_KERNEL();
    return out;
  }
  at::Tensor o_lat = part_o;
  if (part_ml) {
    o_lat = at::empty({R, H, n}, part_o.options());
    latent_decode_merge_kernel<<<dim3((n + LM_COLS - 1) / LM_COLS, H, R), dim3(256),
                                 ((S + 3) / 4 * 4 + 1024) * sizeof(float), stream>>>(
        part_o.data_ptr<float>(), part_ml->data_ptr<float>(), o_lat.data_ptr<float>(), (int)H,
        (int)n, (int)S);
    HIP_CHECK_KERNEL();
  }
  if (wide) {
    latent_decode_value_mfma_kernel<<<dim3((dv + 15) / 16, H, (R + 15) / 16), dim3(256), 0,
                                      stream>>>(
        o_lat.data_ptr<float>(), reinterpret_cast<const bf16*>(w_uv.data_ptr()),
        reinterpret_cast<bf16*>(out.data_ptr()), (int)R, (int)H, (int)dv, (int)rank, (int)n);
    HIP_CHECK_KERNEL();
    return out;
  }
#define LAUNCH(TT, VV)                                                                          \
  latent_decode_value_kernel<TT, VV, RT>                                                        \
      <<<dim3((dv + LC_ROWS - 1) / LC_ROWS, H, (R + RT - 1) / RT), dim3(256), smem, stream>>>(  \
          o_lat.data_ptr<float>(), reinterpret_cast<const TT*>(w_uv.data_ptr()),                \
          reinterpret_cast<TT*>(out.data_ptr()), (int)R, (int)H, (int)dv, (int)rank, (int)n)
  ROW_TILE(R, {
    const size_t smem = RT * rank * sizeof(float);
    TORCH_CHECK(smem <= 64 * 1024, "latent_decode_combine: rank too large");
    if (w_uv.scalar_type() == at::kBFloat16) {
      if (vec) LAUNCH(bf16, 8); else LAUNCH(bf16, 1);
    } else {
      if (vec) LAUNCH(float, 8); else LAUNCH(float, 1);
    }
  });
#undef LAUNCH
  HIP_CHECK_KERNEL();
  return out;
}
#undef ROW_TILE

}  // namespace amd_ops
