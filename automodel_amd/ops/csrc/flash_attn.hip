// Flash attention forward (CDNA4, gfx950): BSHD and packed varlen (THD), causal, GQA,
// head dims {64, 96, 128, 192, 256} and split dims (qk 192 / v 128), optional sinks.
//
// A workgroup takes 32 query rows of one head per wave and walks K/V in tiles of 64 keys,
// double-buffered in LDS by direct loads, one barrier a tile. Both products have the query
// as the accumulator's column, so that a row's maximum, sum and rescaling are per-lane
// values (flash_tile.h).
//
// The products of a tile take 1024 cycles of a SIMD's matrix core and its softmax about
// 900 of the vector unit, so the loop is pipelined over half tiles: while half tile i goes
// through exp, the matrix core forms the scores of i + 1 and the values of i - 1. Two waves
// a SIMD, or two workgroups a CU, fill what one wave leaves. Bound by instruction issue (at
// (128, 128) 96% of the cycles, the matrix core busy 45% and LDS 23% of them, before whole
// tiles had a loop of their own). Long walks of (128, 128) and (192, 128) without documents
// have the kernel of flash_fwd.h.
// Measured (causal, bf16, before -> now): 1 x 16384, 32/8 heads of 128: 6.52 -> 2.02 ms,
// 1090 TFLOP/s (there flash_fwd.h takes 1.84); 2 x 4096: 1030 -> 289 us; 2 x 3072, 16 heads
// (192, 128): 414 -> 120 us; 4 x 2048, 16/8 heads of 64: 154 -> 55 us; 2 x 4096, 8 heads of 256: 544 -> 207 us.
//
// Varlen: per-token doc_start gates the causal mask to the query's own document; tiles
// before a block's first document are skipped.

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <climits>

#include "common.h"
#include "flash_fwd.h"
#include "flash_tile.h"
#include "ops_api.h"

namespace amd_ops {

using namespace fa;

struct FwdArgs {
  const bf16 *q, *k, *v;
  bf16* out;
  float* lse;
  const int* doc_start;
  const bf16* sink;
  int B, Sq, Skv, Hq, Hk, q_start;
  float scale_log2;      // |scale| * log2(e)
  bool negative;         // scale < 0: q changes sign
  bool causal;
};

template <int DQK, int DV, int WAVES, bool VARLEN>
struct Fwd {
  static constexpr int BM = WAVES * 32;
  static constexpr int KT = 64 * row_bytes(DQK), VT = 64 * row_bytes(DV);   // tile bytes
  static constexpr int SMEM = 2 * KT + 2 * VT;
  static constexpr int NC = DQK / 16, NT = DV / 32;

  char* smem;
  unsigned kbase, vbase;
  float c;               // scale * log2(e)
  bf16x8_t qf[NC];
  f32x16_t o[NT];
  float m, l;            // maximum (unscaled) and this half-wave's sum of its row
  int qpos, qdoc, skv;
  bool causal;

  // scores of the 32 keys `sub` of a K tile
  __device__ __forceinline__ void scores(f32x16_t& s, unsigned ktile, int sub) {
    s = zero16();
#pragma unroll
    for (int ch = 0; ch < NC; ++ch) s = mma(read_rows<DQK>(smem, ktile, kbase, sub, ch), qf[ch], s);
  }

  __device__ __forceinline__ void values(const bf16x8_t (&p)[2], unsigned vtile, int sub) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int ch = 0; ch < 2; ++ch)
        o[t] = mma(read_cols<DV>(smem, vtile, vbase, sub, ch, t), p[ch], o[t]);
  }

  // Scores `s` of keys k0.. become probabilities `p`; `meanwhile` holds products that do
  // not depend on them. The maximum is kept while no row grows by more than 2^12 over it:
  // the f32 sums have room for that, and the pass over the output is skipped.
  template <bool MASK, typename Meanwhile>
  __device__ __forceinline__ void softmax(f32x16_t& s, int k0, bf16x8_t (&p)[2], Meanwhile meanwhile) {
    const int half = (threadIdx.x >> 5) & 1;
    if constexpr (MASK) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = k0 + acc_row(r, half);
        const bool dead = (causal && key > qpos) || key >= skv || (VARLEN && key < qdoc);
        s[r] = dead ? -INFINITY : s[r];
      }
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = max_halves(mx);
    const bool rescale = __any((mx - m) * c > 12.f);
    meanwhile();
    const float mn = rescale ? fmaxf(m, mx) : m;
    const float alpha = __builtin_amdgcn_exp2f((m - mn) * c);
    const float mc = mn * c;
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], c, -mc));
      sum += s[r];
    }
    l = l * alpha + sum;
    m = mn;
    p[0] = pack8(s, 0);
    p[1] = pack8(s, 1);
    if (rescale) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] *= alpha;
    }
  }
};

template <int DQK, int DV, int WAVES, int OCC, bool VARLEN>
__global__ __launch_bounds__(64 * WAVES, OCC) void flash_fwd_kernel(const FwdArgs a) {
  using F = Fwd<DQK, DV, WAVES, VARLEN>;
  constexpr int KT = F::KT, VT = F::VT;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  F f;
  f.smem = smem;
  f.kbase = rows_base<DQK>();
  f.vbase = cols_base<DV>();
  f.c = a.scale_log2;
  f.skv = a.Skv;
  f.causal = a.causal;

  const Place at = place_block((a.Sq + F::BM - 1) / F::BM, a.Hq, a.B, a.causal);
  const int half = (threadIdx.x >> 5) & 1, col = threadIdx.x & 31;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = at.head, b = at.batch, kvh = h / (a.Hq / a.Hk);
  const int qblk = at.tile * F::BM;                   // block's, wave's first query row
  const int q0 = qblk + wid * 32;

  const unsigned k_rs = (unsigned)a.Hk * DQK * 2, v_rs = (unsigned)a.Hk * DV * 2;
  const char* kp = reinterpret_cast<const char*>(a.k + ((long)b * a.Skv * a.Hk + kvh) * DQK);
  const char* vp = reinterpret_cast<const char*>(a.v + ((long)b * a.Skv * a.Hk + kvh) * DV);

  {
    const int row = min(q0 + col, a.Sq - 1);          // rows beyond Sq are not stored
    const bf16* src = a.q + (((long)b * a.Sq + row) * a.Hq + h) * DQK + half * 8;
#pragma unroll
    for (int ch = 0; ch < F::NC; ++ch) {
      uint4 w = *reinterpret_cast<const uint4*>(src + ch * 16);
      if (a.negative) {
        w.x ^= 0x80008000u; w.y ^= 0x80008000u; w.z ^= 0x80008000u; w.w ^= 0x80008000u;
      }
      f.qf[ch] = __builtin_bit_cast(bf16x8_t, w);
    }
    f.qpos = a.q_start + q0 + col;
    f.qdoc = VARLEN ? a.doc_start[a.q_start + row] : 0;
    f.m = -1e30f;
    f.l = 0.f;
#pragma unroll
    for (int t = 0; t < F::NT; ++t) f.o[t] = zero16();
  }

  // tiles of the block and of the wave (doc_start does not decrease)
  const int last = a.q_start + min(qblk + F::BM, a.Sq) - 1;
  const int last_w = a.q_start + min(q0 + 32, a.Sq) - 1;
  const int all = (a.Skv + 63) / 64;
  const int t1 = a.causal ? min(last / 64 + 1, all) : all;
  const int t1w = q0 >= a.Sq ? 0 : a.causal ? min(last_w / 64 + 1, all) : all;
  int t0 = 0, t0w = 0, doc_w = 0;
  if (VARLEN) {
    t0 = __builtin_amdgcn_readfirstlane(a.doc_start[a.q_start + qblk]) / 64;
    t0w = __builtin_amdgcn_readfirstlane(a.doc_start[a.q_start + min(q0, a.Sq - 1)]) / 64;
    doc_w = __builtin_amdgcn_readfirstlane(a.doc_start[last_w]);
  }
  // first tile with a key that some row of the wave must not see (from the diagonal on)
  const int t_diag = a.causal ? (a.q_start + q0 + 1) / 64 : all;

  const unsigned lds = lds_address(smem);
  auto load_k = [&](int t) {
    load_tile<DQK, 64, WAVES>(kp + (long)t * 64 * k_rs, k_rs, a.Skv - t * 64, lds + (t & 1) * KT);
  };
  auto load_v = [&](int t) {
    load_tile<DV, 64, WAVES>(vp + (long)t * 64 * v_rs, v_rs, a.Skv - t * 64, lds + 2 * KT + (t & 1) * VT);
  };
  f32x16_t s0, s1;
  bf16x8_t p0[2], p1[2];

  if (t0 < t1) {
    load_k(t0);
    wait_loads();
    barrier();
    if (t0 + 1 < t1) load_k(t0 + 1);
    load_v(t0);
  }
  // A tile that every row of the wave sees whole, with neighbours on both sides: the hot
  // loop, without a branch but the rescaling. At two waves a SIMD instructions are issued
  // nearly all the time, so that each one less counts: one loop with all of a tile's cases
  // kept the output in two sets of registers and moved it between them, and buffers
  // known when this is compiled are offsets in the reads (29 us of the next figure). 16384, 32/8
  // heads of 128: 2499 -> 2187 us; 2 x 3072, 16 heads of (192, 128): 168 -> 120.
  auto steady = [&](int t, auto parity) {
    constexpr int PARITY = decltype(parity)::value;      // of t; -1: any
    const unsigned odd = PARITY < 0 ? t % 2 : PARITY, kt = odd * KT, kn = KT - kt;
    const unsigned vt = 2 * KT + odd * VT, vo = 4 * KT + VT - vt;
    f.template softmax<false>(s0, t * 64, p0, [&] { f.scores(s1, kt, 1); f.values(p1, vo, 1); });
    wait_loads();       // K of t + 1, V of t; the buffers of K of t, V of t - 1 are free
    barrier();
    load_v(t + 1);
    load_k(t + 2);
    f.template softmax<false>(s1, t * 64 + 32, p1, [&] { f.scores(s0, kn, 0); f.values(p0, vt, 0); });
  };
  auto general = [&](int t) {
    const bool live = t >= t0w && t < t1w;
    const unsigned kt = (t & 1) * KT, kn = KT - kt;
    const unsigned vt = 2 * KT + (t & 1) * VT, vo = 4 * KT + VT - vt;
    if (live) {
      if (t == t0w) f.scores(s0, kt, 0);
      f.template softmax<true>(s0, t * 64, p0, [&] {
        f.scores(s1, kt, 1);
        if (t != t0w) f.values(p1, vo, 1);
      });
    }
    wait_loads();
    barrier();
    if (t + 1 < t1) load_v(t + 1);
    if (t + 2 < t1) load_k(t + 2);
    if (live) {
      // (the scores of the tile after a wave's last one are formed and not used)
      f.template softmax<true>(s1, t * 64 + 32, p1, [&] { f.scores(s0, kn, 0); f.values(p0, vt, 0); });
      if (t == t1w - 1) f.values(p1, vt, 1);
    }
  };
  // Tiles of the steady kind: [first, end). There is a tile t + 2 for each of them to load:
  // the buffer of t + 1, which a step reads, has no load in flight.
  const int first = max(t0w + 1, VARLEN ? (doc_w + 63) / 64 : 0);
  const int end = min(min(t_diag, a.Skv / 64), min(t1w - 1, t1 - 2));
  // Pairs leave a tile over at either end: the runs of short documents are too short for
  // them. With 256 columns of output they spill; one at a time does not (2 x 4096 tokens, 8
  // heads of 256: 207 us, 494 with scores, softmax and values one after the other, 544 with the
  // kernel before; without a mask 378, 895 and 558).
  constexpr bool PAIRS = !VARLEN && DV < 256;
  int t = t0;
  for (; t < min(first, t1) || (PAIRS && t < end && t % 2); ++t) general(t);
  if constexpr (!PAIRS)
    for (; t < end; ++t) steady(t, std::integral_constant<int, -1>{});
  else
    for (; t + 1 < end; t += 2) {
      steady(t, std::integral_constant<int, 0>{});
      steady(t + 1, std::integral_constant<int, 1>{});
    }
  for (; t < t1; ++t) general(t);

  // ---- normalise, then through LDS (the tiles are done with) to whole-row stores. A
  // sink is one more logit in the denominator, without a key.
  constexpr int RB = row_bytes(DV);
  static_assert(F::SMEM >= F::BM * RB, "output tile fits the K/V buffers");
  barrier();
  char* mine = smem + wid * 32 * RB;
  const float l = sum_halves(f.l), m2 = f.m * f.c;    // maximum in units of log2
  const float ls = a.sink ? l + __builtin_amdgcn_exp2f(bf2f(a.sink[h]) * LOG2E - m2) : l;
  const float inv = ls > 0.f ? 1.f / ls : 0.f;
  if (half == 0 && q0 + col < a.Sq)
    a.lse[((long)b * a.Hq + h) * a.Sq + q0 + col] = ls > 0.f ? m2 * LN2 + __logf(ls) : -1e30f;
  store_rows<DV>(f.o, inv, mine, a.out + (((long)b * a.Sq + q0) * a.Hq + h) * DV, (long)a.Hq * DV,
                 a.Sq - q0);
}

// document [start, end) of every token of a packed row, by bisection of cu; what lies
// beyond cu's last entry is a document of its own
__global__ void doc_bounds_kernel(const int* __restrict__ cu, int n, int total, int* __restrict__ start,
                                  int* __restrict__ end) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= total) return;
  int lo = 0, hi = n;                   // first entry greater than t
  while (lo < hi) {
    const int mid = (lo + hi) / 2;
    if (cu[mid] > t) hi = mid; else lo = mid + 1;
  }
  start[t] = lo > 0 ? cu[lo - 1] : 0;
  end[t] = lo < n ? cu[lo] : total;
}

std::tuple<at::Tensor, at::Tensor> doc_bounds(const at::Tensor& cu, int64_t total) {
  TORCH_CHECK(cu.is_cuda() && cu.dim() == 1 && cu.scalar_type() == at::kInt && cu.is_contiguous() &&
                  cu.numel() >= 1 && total >= 0, "doc_bounds: cu_seqlens int32 [n + 1]");
  auto start = at::empty({total}, cu.options()), end = at::empty({total}, cu.options());
  if (total == 0) return {start, end};
  hipLaunchKernelGGL(doc_bounds_kernel, dim3(ceil_div_i(total, 256)), dim3(256), 0,
                     c10::hip::getCurrentHIPStream().stream(), cu.data_ptr<int>(), (int)cu.numel(),
                     (int)total, start.data_ptr<int>(), end.data_ptr<int>());
  HIP_CHECK_KERNEL();
  return {start, end};
}

template <int DQK, int DV, int WAVES, int OCC, bool VARLEN>
static void launch_fwd(const FwdArgs& a, hipStream_t stream) {
  using F = Fwd<DQK, DV, WAVES, VARLEN>;
  const long blocks = (long)((a.Sq + F::BM - 1) / F::BM) * a.Hq * a.B;
  hipLaunchKernelGGL((flash_fwd_kernel<DQK, DV, WAVES, OCC, VARLEN>), dim3((unsigned)blocks),
                     dim3(64 * WAVES), F::SMEM, stream, a);
  HIP_CHECK_KERNEL();
}

template <int DQK, int DV, int N>
static void launch_fwd_ordered(const FwdArgs& a, hipStream_t stream) {
  using T = FwdTile<DQK, DV, N>;
  const long blocks = (long)((a.Sq + T::BM - 1) / T::BM) * a.Hq * a.B;
  hipLaunchKernelGGL((flash_fwd_ordered_kernel<DQK, DV, N, FwdArgs>), dim3((unsigned)blocks), dim3(256), T::SMEM,
                     stream, a);
  HIP_CHECK_KERNEL();
}

template <int N>
static long ordered_blocks(const FwdArgs& a) { return (long)((a.Sq + 64 * N - 1) / (64 * N)) * a.Hq * a.B; }

// Sixteens of rows a wave of the kernel in a given order, or 0: the one above. Times in us, the kernel above
// first; batch x length, heads.
//
// (128, 128): a workgroup has 256 rows and a CU, against 128 and half of one. Without a mask it wants
// full rounds of workgroups, counted in rows, as the last workgroup of a sequence may be nearly empty (1 x 8192,
// 8: 264 and 228; 8 x 1024, 32: 179 and 156; 2 x 1024, 32: 42.5 and 42.3; but 1 x 5000, 32, two and a half
// rounds: 406 and 424; 1672, 128 in all, 0.82 of four: 222 and 250; 4 x 512, 32: 27.5 and 28.6). With a causal
// one, whose last tiles are wasted on most waves, long rows, and two rounds (1 x 8000, 16: 277 and 251;
// 1 x 16384, 32: 2020 and 1843; but 2 x 6000, 16: 294 and 304; 1 x 8192, 8: 183 and 228). Few queries
// leave its waves empty rows (8 x 64 of 4096 keys, 32: 102 and 134).
static int ordered_rows_128(const FwdArgs& a) {
  if (a.Sq < 1024) return 0;
  const long blocks = ordered_blocks<4>(a), rounds = (blocks + 255) / 256;
  if (a.causal) return a.Skv >= 8000 && blocks >= 512 ? 4 : 0;
  return a.Skv >= 1024 && (double)a.Sq * a.Hq * a.B >= 0.85 * 65536 * rounds ? 4 : 0;
}

// (192, 128): 4 sixteens against 3, which take 0.77 of the time of 4: by rounds of workgroups without a
// mask (2 x 3001, 16: 164 against 201; 2 x 2048, 16: 111 against 77), with a causal one by the longest
// workgroup or all of them, what is more (2 x 3001, 16: 98 against 103; 1 x 8192, 16: 325 against 292).
// The kernel above has 8 waves for 256 rows: it stays for short rows (1 x 100, 4: 9.1 and 12.8; without a
// mask 4 x 512, 32: 32.7 and 33.9), and, where each workgroup has few tiles and wasted ones among them,
// with a causal mask (16 x 1500, 32: 560 and 593; 2 x 1024, 32: 44.2 and 47.6; but 1 x 1024, 32, one
// round: 41.5 and 34.6; 2 x 2048, 16: 72 and 57; 2 x 4096, 32: 356 and 338); and for fewer queries than a
// workgroup's (8 x 64 of 4096 keys, 32: 119 and 129; 1 x 192 of 8192, 16: 239 and 189).
static int ordered_rows_192(const FwdArgs& a) {
  if (a.Sq < 192) return 0;
  const long b4 = ordered_blocks<4>(a), b3 = ordered_blocks<3>(a);
  if (!a.causal) {
    if ((b3 + 255) / 256 * 0.77 < (double)((b4 + 255) / 256)) return a.Skv >= 512 ? 3 : 0;
    return a.Skv >= 1024 ? 4 : 0;
  }
  const double longest = std::min<long>((long)a.q_start + a.Sq, a.Skv);
  // the workgroups in the order of their lengths, the longest first: the two that follow one another on
  // a CU are about as long together everywhere, and of an odd number of rounds the last one begins with its
  // longest (3465, 32 in all: 608 workgroups of 192 rows, 170 us, 150 the kernel above, 149 in fours)
  auto cost = [&](long blocks, int rows) {
    const double first = std::min<long>((long)a.q_start + rows, a.Skv), all = blocks * (longest + first) / 2;
    const long k = (blocks + 255) / 256, pairs = k / 2 * 2;
    if (k == 1) return longest;
    const double before = pairs * (256. * pairs - 1) / 2 + (k > pairs ? 256. * pairs : 0.);
    return std::max({longest, all / 256, k * longest - (longest - first) * before / (blocks - 1)});
  };
  const double c4 = cost(b4, 256), c3 = cost(b3, 192) * 0.77;
  if (a.Skv >= 3000) return c3 < c4 ? 3 : 4;
  return (a.Skv >= 512 && b3 <= 256) || (a.Skv >= 2048 && c3 < 0.9 * c4) ? 3 : 0;
}

// of any dims, without documents
static int ordered_rows(const FwdArgs& a, int Dqk, int Dv) {
  if (Dv != 128 || (Dqk != 128 && Dqk != 192)) return 0;
  return Dqk == 128 ? ordered_rows_128(a) : ordered_rows_192(a);
}

int64_t flash_attn_fwd_ordered(int64_t B, int64_t Sq, int64_t Skv, int64_t Hq, int64_t Hk, int64_t Dqk, int64_t Dv,
                               bool causal, int64_t q_start) {
  TORCH_CHECK(std::min({B, Sq, Skv, Hq, Hk}) >= 1 && std::max({B, Sq, Skv, Hq, Hk, q_start}) <= INT_MAX &&
                  Hq % Hk == 0 && q_start >= 0, "flash_attn_fwd_ordered: sizes");
  FwdArgs a{};
  a.B = (int)B; a.Sq = (int)Sq; a.Skv = (int)Skv; a.Hq = (int)Hq; a.Hk = (int)Hk; a.q_start = (int)q_start;
  a.causal = causal;
  return ordered_rows(a, (int)Dqk, (int)Dv);
}

std::tuple<at::Tensor, at::Tensor> flash_attn_fwd(
    const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, double scale,
    bool causal, int64_t q_start, const std::optional<at::Tensor>& doc_start,
    const std::optional<at::Tensor>& sink) {
  TORCH_CHECK(q.is_cuda() && q.dim() == 4 && q.scalar_type() == at::kBFloat16,
              "flash_attn_fwd: q must be [B,S,Hq,D] bf16");
  const int B = q.size(0), Sq = q.size(1), Hq = q.size(2), Dqk = q.size(3);
  const int Skv = k.size(1), Hk = k.size(2), Dv = v.size(3);
  TORCH_CHECK(Hq % Hk == 0, "flash_attn_fwd: Hq must be divisible by Hk");
  TORCH_CHECK(k.size(0) == B && v.size(0) == B && k.size(3) == Dqk && v.size(1) == Skv && v.size(2) == Hk &&
                  q.is_contiguous() && k.is_contiguous() && v.is_contiguous(),
              "flash_attn_fwd: contiguous k [B,Skv,Hk,Dqk], v [B,Skv,Hk,Dv]");
  TORCH_CHECK(Sq >= 1 && Skv >= 1, "flash_attn_fwd: empty sequences");
  const bool varlen = doc_start.has_value();
  if (varlen)
    TORCH_CHECK(doc_start->numel() >= q_start + Sq, "flash_attn_fwd: doc_start for every query position");
  if (varlen) TORCH_CHECK(causal && B == 1, "varlen flash is causal with B==1");
  if (sink)
    TORCH_CHECK(sink->is_cuda() && sink->is_contiguous() && sink->numel() == Hq &&
                    sink->scalar_type() == at::kBFloat16, "flash_attn_fwd: sink [Hq] bf16");
  auto out = at::empty({B, Sq, Hq, Dv}, q.options());
  auto lse = at::empty({B, Hq, Sq}, q.options().dtype(at::kFloat));
  auto stream = c10::hip::getCurrentHIPStream().stream();
  FwdArgs a;
  a.q = reinterpret_cast<const bf16*>(q.data_ptr());
  a.k = reinterpret_cast<const bf16*>(k.data_ptr());
  a.v = reinterpret_cast<const bf16*>(v.data_ptr());
  a.out = reinterpret_cast<bf16*>(out.data_ptr());
  a.lse = lse.data_ptr<float>();
  a.doc_start = varlen ? doc_start->data_ptr<int>() : nullptr;
  a.sink = sink ? reinterpret_cast<const bf16*>(sink->data_ptr()) : nullptr;
  a.B = B; a.Sq = Sq; a.Skv = Skv; a.Hq = Hq; a.Hk = Hk; a.q_start = (int)q_start;
  // a scale of zero: equal weights, whatever the scores (masked ones stay masked)
  a.scale_log2 = std::max((float)std::fabs(scale) * LOG2E, 1e-37f);
  a.negative = scale < 0;
  a.causal = causal;

  // Waves per workgroup and per SIMD: as many as the registers of the accumulators and
  // the two K/V tiles in LDS allow. (192, 128) fits one workgroup a CU, so it has 8 waves
  // (120 us; 4 waves at one a SIMD were 1.3 times slower); (192, 192) would spill at two a SIMD (457
  // against 178 us).
  bool done = false;
  if (const int n = varlen ? 0 : ordered_rows(a, Dqk, Dv); n > 0) {
    done = true;
    if (Dqk == 128) launch_fwd_ordered<128, 128, 4>(a, stream);
    else if (n == 4) launch_fwd_ordered<192, 128, 4>(a, stream);
    else launch_fwd_ordered<192, 128, 3>(a, stream);
  }
#define FA_FWD_CASE(A, C, W, OCC)                             \
  if (!done && Dqk == A && Dv == C) {                         \
    done = true;                                              \
    if (varlen) launch_fwd<A, C, W, OCC, true>(a, stream);    \
    else launch_fwd<A, C, W, OCC, false>(a, stream);          \
  }
  FA_FWD_CASE(64, 64, 4, 3)
  FA_FWD_CASE(96, 96, 4, 2)
  FA_FWD_CASE(128, 128, 4, 2)
  FA_FWD_CASE(192, 128, 8, 2)
  FA_FWD_CASE(192, 192, 4, 1)
  FA_FWD_CASE(256, 256, 4, 1)
#undef FA_FWD_CASE
  TORCH_CHECK(done, "flash_attn_fwd: unsupported head dims (Dqk=", Dqk, ", Dv=", Dv,
              "); supported pairs: (64,64),(96,96),(128,128),(192,128),(192,192),(256,256)");
  return {out, lse};
}

}  // namespace amd_ops
