// Attention of one new token per sequence over the dense K/V cache
// [B, max_len, Hk, D], and the cache write of that token.
//
// Bound by reading the cache once. A row of K or V lies over LPK lanes of 16 bytes, a wave
// loads 64 / LPK keys at a time straight into registers and works on 4 such loads of each
// per iteration; the GQ query heads that share the K/V head are all served from them. The
// dot products are vector instructions: with a handful of queries a matrix instruction
// would be empty for the most part, and a key costs a CU about 25 cycles against the 65
// that its 512 bytes (head dim 128) take from memory. Every lane group keeps maximum, sum
// and output of its own keys, so that the loop needs no exchange beyond the row sums (DPP);
// groups, waves and splits are merged at the end. Everything is f32 except the cache.
//
// The sequence is cut into splits until some 1024 workgroups are in flight; the position is
// a host number or, for captured steps, a device counter (splits then follow the cache's
// capacity, and their borders the counter). The new token's K and V come from the call's
// own tensors, and the workgroup of their split stores them: no workgroup reads what
// another one writes.
//
// Measured, 32/8 heads of 128, with merge: 16 x 1500 keys 31 us, 1 x 512 11 us, 32 x 4096 120 us
// (4.5 TB/s); the chain of mask, casts, repeats and f32 products before took 0.71 ms and 0.08 ms
// for the first two.

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include "common.h"
#include "ops_api.h"

namespace amd_ops {

namespace {

constexpr float LOG2E_F = 1.4426950408889634f;
constexpr int UNROLL = 4;              // loads of K and of V in flight per lane

template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, false));
}
// sum over the LPK lanes (8, 16 or 32) that hold one key
template <int LPK>
__device__ __forceinline__ float key_sum(float x) {
  x = dpp_add<0xB1>(x);                // quad_perm: lane ^ 1
  x = dpp_add<0x4E>(x);                // quad_perm: lane ^ 2
  x = dpp_add<0x141>(x);               // mirror within 8
  if constexpr (LPK >= 16) x = dpp_add<0x140>(x);      // mirror within 16
  if constexpr (LPK >= 32) x += __shfl_xor(x, 16);
  return x;
}

__device__ __forceinline__ void unpack8(const uint4& w, float (&f)[8]) {
  const unsigned u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = __uint_as_float(u[i] << 16);
    f[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
  }
}

struct KvArgs {
  const bf16 *q, *k_new, *v_new;
  bf16 *k_cache, *v_cache, *out;
  float *part_o, *part_ml;
  const long* pos_dev;
  long batch_stride;                   // of the caches, in elements
  int pos, max_len, Hq, Hk, D, splits;
  float scale_log2;
};

}  // namespace

template <int LPK, int GQ>
__global__ __launch_bounds__(256) void kv_decode_kernel(const KvArgs a) {
  constexpr int KPW = 64 / LPK, STEP = 4 * KPW * UNROLL;       // keys per load, per iteration
  __shared__ __attribute__((aligned(16))) float so[4][GQ][LPK * 8];
  __shared__ float sm[4][GQ], sl[4][GQ];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int l = lane % LPK, kg = lane / LPK;
  const int split = blockIdx.x, b = blockIdx.z;
  const int group = a.Hq / a.Hk, chunks = (group + GQ - 1) / GQ;
  const int kvh = blockIdx.y / chunks, g0 = blockIdx.y % chunks * GQ;
  const int pos = a.pos_dev ? (int)min(a.pos_dev[0], (long)a.max_len - 1) : a.pos;
  const int D = a.D, row = a.Hk * D;
  const bool lane_in = l * 8 < D;

  // whole iterations per split; the last one may be short, later ones empty
  const int len = pos + 1;
  const int per = ((len + a.splits - 1) / a.splits + STEP - 1) / STEP * STEP;
  const int k0 = split * per, k1 = min(k0 + per, len);

  const long head = (long)kvh * D + l * 8;
  bf16* kc = a.k_cache + (long)b * a.batch_stride + head;
  bf16* vc = a.v_cache + (long)b * a.batch_stride + head;
  const long at_new = (long)b * row + head;

  float q[GQ][8], o[GQ][8], m[GQ], s_sum[GQ];
#pragma unroll
  for (int g = 0; g < GQ; ++g) {
    const int h = kvh * group + min(g0 + g, group - 1);       // (heads beyond the group: not stored)
    uint4 w = {0, 0, 0, 0};
    if (lane_in) w = *reinterpret_cast<const uint4*>(a.q + ((long)b * a.Hq + h) * D + l * 8);
    unpack8(w, q[g]);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      q[g][j] *= a.scale_log2;
      o[g][j] = 0.f;
    }
    m[g] = -1e30f;
    s_sum[g] = 0.f;
  }

  for (int kb = k0; kb < k1; kb += STEP) {
    uint4 kw[UNROLL], vw[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int key = kb + (u * 4 + wid) * KPW + kg;
      kw[u] = vw[u] = {0, 0, 0, 0};
      if (lane_in && key < k1) {
        // the token of this call is in its own tensors, not yet in the cache
        const bf16* kp = key == pos ? a.k_new + at_new : kc + (long)key * row;
        const bf16* vp = key == pos ? a.v_new + at_new : vc + (long)key * row;
        kw[u] = *reinterpret_cast<const uint4*>(kp);
        vw[u] = *reinterpret_cast<const uint4*>(vp);
        if (key == pos && g0 == 0) {
          *reinterpret_cast<uint4*>(kc + (long)key * row) = kw[u];
          *reinterpret_cast<uint4*>(vc + (long)key * row) = vw[u];
        }
      }
    }
    float s[UNROLL][GQ];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      float kf[8];
      unpack8(kw[u], kf);
      const bool in = kb + (u * 4 + wid) * KPW + kg < k1;
#pragma unroll
      for (int g = 0; g < GQ; ++g) {
        float t = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) t = fmaf(q[g][j], kf[j], t);
        t = key_sum<LPK>(t);
        s[u][g] = in ? t : -INFINITY;
      }
    }
#pragma unroll
    for (int g = 0; g < GQ; ++g) {
      float mn = m[g];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) mn = fmaxf(mn, s[u][g]);
      const float alpha = __builtin_amdgcn_exp2f(m[g] - mn);
      m[g] = mn;
      s_sum[g] *= alpha;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[g][j] *= alpha;
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        s[u][g] = __builtin_amdgcn_exp2f(s[u][g] - mn);
        s_sum[g] += s[u][g];
      }
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      float vf[8];
      unpack8(vw[u], vf);
#pragma unroll
      for (int g = 0; g < GQ; ++g)
#pragma unroll
        for (int j = 0; j < 8; ++j) o[g][j] = fmaf(s[u][g], vf[j], o[g][j]);
    }
  }

  // lane groups of the wave, then the waves
#pragma unroll
  for (int g = 0; g < GQ; ++g) {
    float mw = m[g];
#pragma unroll
    for (int off = LPK; off < 64; off <<= 1) mw = fmaxf(mw, __shfl_xor(mw, off));
    const float f = __builtin_amdgcn_exp2f(m[g] - mw);
    s_sum[g] *= f;
#pragma unroll
    for (int off = LPK; off < 64; off <<= 1) s_sum[g] += __shfl_xor(s_sum[g], off);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      o[g][j] *= f;
#pragma unroll
      for (int off = LPK; off < 64; off <<= 1) o[g][j] += __shfl_xor(o[g][j], off);
    }
    if (kg == 0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) so[wid][g][l * 8 + j] = o[g][j];
      if (l == 0) {
        sm[wid][g] = mw;
        sl[wid][g] = s_sum[g];
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < GQ * D; i += 256) {
    const int g = i / D, d = i % D;
    if (g0 + g >= group) break;
    const long h = (long)b * a.Hq + kvh * group + g0 + g;
    const float mx = fmaxf(fmaxf(sm[0][g], sm[1][g]), fmaxf(sm[2][g], sm[3][g]));
    float acc = 0.f, sum = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = __builtin_amdgcn_exp2f(sm[w][g] - mx);
      acc = fmaf(so[w][g][d], f, acc);
      sum = fmaf(sl[w][g], f, sum);
    }
    if (a.splits == 1) {
      a.out[h * D + d] = f2bf(acc / sum);
    } else {
      a.part_o[(h * a.splits + split) * D + d] = acc;
      if (d == 0) {
        a.part_ml[(h * a.splits + split) * 2] = mx;
        a.part_ml[(h * a.splits + split) * 2 + 1] = sum;
      }
    }
  }
}

// splits (at most 64) of one head -> output: a lane per split for the weights, then a
// thread per column
__global__ __launch_bounds__(256) void kv_decode_merge_kernel(const float* __restrict__ part_o,
                                                              const float* __restrict__ part_ml,
                                                              bf16* __restrict__ out, int splits,
                                                              int D) {
  __shared__ float w[64];
  const long h = blockIdx.x;
  if (threadIdx.x < 64) {
    const int i = threadIdx.x;
    const float m = i < splits ? part_ml[(h * splits + i) * 2] : -1e30f;
    const float s = i < splits ? part_ml[(h * splits + i) * 2 + 1] : 0.f;
    const float f = __builtin_amdgcn_exp2f(m - wave_reduce_max(m));
    const float sum = wave_reduce_sum(s * f);
    w[i] = f / sum;
  }
  __syncthreads();
  for (int d = threadIdx.x; d < D; d += blockDim.x) {
    float acc = 0.f;
#pragma unroll 8
    for (int i = 0; i < splits; ++i) acc = fmaf(part_o[(h * splits + i) * D + d], w[i], acc);
    out[h * D + d] = f2bf(acc);
  }
}

at::Tensor kv_decode_attn(const at::Tensor& q, const at::Tensor& k_new, const at::Tensor& v_new,
                          at::Tensor k_cache, at::Tensor v_cache, int64_t pos,
                          const std::optional<at::Tensor>& pos_dev, double scale) {
  TORCH_CHECK(q.is_cuda() && q.dim() == 4 && q.size(1) == 1 && q.scalar_type() == at::kBFloat16 &&
                  q.is_contiguous(), "kv_decode_attn: q [B,1,Hq,D] bf16");
  const int B = q.size(0), Hq = q.size(2), D = q.size(3);
  TORCH_CHECK(k_cache.dim() == 4 && k_cache.scalar_type() == at::kBFloat16 && k_cache.is_contiguous() &&
                  v_cache.sizes() == k_cache.sizes() && v_cache.scalar_type() == at::kBFloat16 &&
                  v_cache.is_contiguous() && k_cache.size(0) >= B && k_cache.size(3) == D,
              "kv_decode_attn: caches [B,max_len,Hk,D] bf16");
  const int max_len = k_cache.size(1), Hk = k_cache.size(2);
  const std::vector<int64_t> one{B, 1, Hk, D};
  TORCH_CHECK(k_new.sizes() == at::IntArrayRef(one) && v_new.sizes() == at::IntArrayRef(one) && k_new.is_contiguous() &&
                  v_new.is_contiguous() && k_new.scalar_type() == at::kBFloat16 &&
                  v_new.scalar_type() == at::kBFloat16, "kv_decode_attn: new k, v [B,1,Hk,D] bf16");
  TORCH_CHECK(Hq % Hk == 0 && D % 8 == 0 && D >= 8 && D <= 256 && B >= 1 && B <= 65535,
              "kv_decode_attn: whole groups, head dim a multiple of 8 up to 256");
  TORCH_CHECK(pos_dev ? pos_dev->device() == q.device() && pos_dev->scalar_type() == at::kLong && pos_dev->numel() == 1
                      : pos >= 0 && pos < max_len, "kv_decode_attn: position outside the cache");
  for (const at::Tensor* t : {&q, &k_new, &v_new, (const at::Tensor*)&k_cache, (const at::Tensor*)&v_cache}) {
    TORCH_CHECK(t->device() == q.device(), "kv_decode_attn: one device");
    TORCH_CHECK((uintptr_t)t->data_ptr() % 16 == 0, "kv_decode_attn: 16-byte alignment");
  }

  const int group = Hq / Hk;
  const int gq = group >= 5 ? 8 : group >= 3 ? 4 : group;
  const int chunks = (group + gq - 1) / gq;
  const int lpk = D <= 64 ? 8 : D <= 128 ? 16 : 32, step = 4 * (64 / lpk) * UNROLL;
  const int len = pos_dev ? max_len : (int)pos + 1;
  const int splits = std::max(1, std::min({1024 / (B * Hk * chunks), (len + step - 1) / step, 64}));

  auto out = at::empty({B, 1, Hq, D}, q.options());
  at::Tensor part;
  KvArgs a;
  a.q = reinterpret_cast<const bf16*>(q.data_ptr());
  a.k_new = reinterpret_cast<const bf16*>(k_new.data_ptr());
  a.v_new = reinterpret_cast<const bf16*>(v_new.data_ptr());
  a.k_cache = reinterpret_cast<bf16*>(k_cache.data_ptr());
  a.v_cache = reinterpret_cast<bf16*>(v_cache.data_ptr());
  a.out = reinterpret_cast<bf16*>(out.data_ptr());
  a.part_o = a.part_ml = nullptr;
  if (splits > 1) {
    part = at::empty({(long)B * Hq * splits * (D + 2)}, q.options().dtype(at::kFloat));
    a.part_o = part.data_ptr<float>();
    a.part_ml = a.part_o + (long)B * Hq * splits * D;
  }
  a.pos_dev = pos_dev ? pos_dev->data_ptr<long>() : nullptr;
  a.batch_stride = (long)max_len * Hk * D;
  a.pos = (int)pos; a.max_len = max_len; a.Hq = Hq; a.Hk = Hk; a.D = D; a.splits = splits;
  a.scale_log2 = (float)scale * LOG2E_F;
  auto stream = c10::hip::getCurrentHIPStream().stream();
  const dim3 grid(splits, Hk * chunks, B);
#define KV_CASE(L, G)                                                                  \
  if (lpk == L && gq == G) {                                                           \
    hipLaunchKernelGGL((kv_decode_kernel<L, G>), grid, dim3(256), 0, stream, a);       \
  }
  KV_CASE(8, 1) KV_CASE(8, 2) KV_CASE(8, 4) KV_CASE(8, 8)
  KV_CASE(16, 1) KV_CASE(16, 2) KV_CASE(16, 4) KV_CASE(16, 8)
  KV_CASE(32, 1) KV_CASE(32, 2) KV_CASE(32, 4) KV_CASE(32, 8)
#undef KV_CASE
  HIP_CHECK_KERNEL();
  if (splits > 1) {
    hipLaunchKernelGGL(kv_decode_merge_kernel, dim3(B * Hq), dim3(D <= 64 ? 64 : D <= 128 ? 128 : 256), 0,
                       stream, a.part_o, a.part_ml, a.out, splits, D);
    HIP_CHECK_KERNEL();
  }
  return out;
}

}  // namespace amd_ops
