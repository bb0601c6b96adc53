// Fused rotary embedding for q and k (CDNA4).
// HF rotate-half convention: y1 = x1*cos - x2*sin ; y2 = x2*cos + x1*sin over
// the two halves of head_dim. cos/sin tables are host-precomputed fp32
// (guide Appendix B: no device trig). One launch covers q AND k.
// Replaces the reference's TE/Liger fused-RoPE backends.

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include "common.h"
#include "ops_api.h"

namespace amd_ops {

// Each thread handles TWO adjacent pairs (4B loads from each half-row).
// rows = B*S*Hq followed by B*S*Hk; table row = s = (flat_row / H) % S.
__global__ void rope_kernel(const bf16* __restrict__ q, const bf16* __restrict__ k,
                            const float* __restrict__ cosb, const float* __restrict__ sinb,
                            bf16* __restrict__ qo, bf16* __restrict__ ko,
                            int S, int Hq, int Hk, int D, long q_rows, long total_rows,
                            float sign) {
  const int half = D / 2;
  const int pairs2 = half / 2;  // 2-pair work items per row
  const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long row = gid / pairs2;
  if (row >= total_rows) return;
  const int p2 = (int)(gid % pairs2);
  const int j = p2 * 2;

  const bf16* src;
  bf16* dst;
  long r;
  int H;
  if (row < q_rows) {
    r = row; H = Hq; src = q; dst = qo;
  } else {
    r = row - q_rows; H = Hk; src = k; dst = ko;
  }
  const int s = (int)((r / H) % S);
  const long base = r * (long)D;

  // 4-byte vector loads: two bf16 from each half
  ushort2 x1u = *reinterpret_cast<const ushort2*>(src + base + j);
  ushort2 x2u = *reinterpret_cast<const ushort2*>(src + base + j + half);
  float2 c = *reinterpret_cast<const float2*>(cosb + (long)s * D + j);
  float2 sn = *reinterpret_cast<const float2*>(sinb + (long)s * D + j);
  sn.x *= sign; sn.y *= sign;

  bf16 x1a = *reinterpret_cast<bf16*>(&x1u.x), x1b = *reinterpret_cast<bf16*>(&x1u.y);
  bf16 x2a = *reinterpret_cast<bf16*>(&x2u.x), x2b = *reinterpret_cast<bf16*>(&x2u.y);
  float f1a = bf2f(x1a), f1b = bf2f(x1b), f2a = bf2f(x2a), f2b = bf2f(x2b);

  bf16 y1a = f2bf(f1a * c.x - f2a * sn.x);
  bf16 y1b = f2bf(f1b * c.y - f2b * sn.y);
  bf16 y2a = f2bf(f2a * c.x + f1a * sn.x);
  bf16 y2b = f2bf(f2b * c.y + f1b * sn.y);

  ushort2 y1u{*reinterpret_cast<unsigned short*>(&y1a), *reinterpret_cast<unsigned short*>(&y1b)};
  ushort2 y2u{*reinterpret_cast<unsigned short*>(&y2a), *reinterpret_cast<unsigned short*>(&y2b)};
  *reinterpret_cast<ushort2*>(dst + base + j) = y1u;
  *reinterpret_cast<ushort2*>(dst + base + j + half) = y2u;
}

// 8 columns of the lower half of a row and the 8 that are rotated with them
__device__ __forceinline__ void rotate8(bf16x8& x1, bf16x8& x2, const float* cos, const float* sin, float sign) {
  float cs[8], sn[8];
#pragma unroll
  for (int j = 0; j < 8; j += 4) {
    *reinterpret_cast<float4*>(cs + j) = *reinterpret_cast<const float4*>(cos + j);
    *reinterpret_cast<float4*>(sn + j) = *reinterpret_cast<const float4*>(sin + j);
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float a = bf2f(x1.v[j]), b = bf2f(x2.v[j]), s = sign * sn[j];
    x1.v[j] = f2bf(fmaf(a, cs[j], -(b * s)));              // (as the compiler has it above: the same bits)
    x2.v[j] = f2bf(fmaf(b, cs[j], a * s));
  }
}

// The kernel above with 16 bytes a load, for heads of a multiple of 16 columns whose tensors lie on such boundaries:
// 8192 rows of 32 + 8 heads of 128 25 us, 36 with 4 bytes a load.
__global__ __launch_bounds__(256) void rope_wide_kernel(const bf16* __restrict__ q, const bf16* __restrict__ k,
                                                        const float* __restrict__ cosb, const float* __restrict__ sinb,
                                                        bf16* __restrict__ qo, bf16* __restrict__ ko, int S, int Hq, int Hk,
                                                        int D, long q_rows, long items, float sign) {
  const long id = (long)blockIdx.x * 256 + threadIdx.x;
  if (id >= items) return;
  const int chunks = D / 16, c = (int)(id % chunks) * 8;
  const long row = id / chunks;
  const bool is_q = row < q_rows;
  const long r = is_q ? row : row - q_rows, at = r * D + c, s = r / (is_q ? Hq : Hk) % S;
  const bf16* from = (is_q ? q : k) + at;
  bf16* to = (is_q ? qo : ko) + at;
  bf16x8 x1 = *reinterpret_cast<const bf16x8*>(from), x2 = *reinterpret_cast<const bf16x8*>(from + D / 2);
  rotate8(x1, x2, cosb + s * D + c, sinb + s * D + c, sign);
  *reinterpret_cast<bf16x8*>(to) = x1;
  *reinterpret_cast<bf16x8*>(to + D / 2) = x2;
}

// q: [B,S,Hq,D] bf16, k: [B,S,Hk,D] bf16, cos/sin: [S,D] f32.
std::tuple<at::Tensor, at::Tensor> rope_fwd(const at::Tensor& q, const at::Tensor& k,
                                            const at::Tensor& cosb, const at::Tensor& sinb,
                                            bool backward) {
  TORCH_CHECK(q.is_cuda() && q.dim() == 4 && q.scalar_type() == at::kBFloat16,
              "rope_fwd: q must be 4-D bf16");
  TORCH_CHECK(cosb.scalar_type() == at::kFloat && cosb.dim() == 2, "rope: cos must be [S,D] f32");
  const int B = q.size(0), S = q.size(1), Hq = q.size(2), D = q.size(3);
  const int Hk = k.size(2);
  TORCH_CHECK(cosb.size(0) >= S && cosb.size(1) == D, "rope: table shape mismatch");
  TORCH_CHECK(D % 4 == 0, "rope: head_dim must be a multiple of 4");
  auto qo = at::empty_like(q);
  auto ko = at::empty_like(k);
  const long q_rows = (long)B * S * Hq;
  const long total_rows = q_rows + (long)B * S * Hk;
  const long work = total_rows * (D / 4);
  const int block = 256;
  const long grid = (work + block - 1) / block;
  auto stream = c10::hip::getCurrentHIPStream();
  bool wide = D % 16 == 0 && total_rows > 0;
  for (const at::Tensor* t : {&q, &k, &cosb, &sinb}) wide = wide && (uintptr_t)t->data_ptr() % 16 == 0;
  if (wide) {
    const long items = total_rows * (D / 16);
    hipLaunchKernelGGL(rope_wide_kernel, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, stream.stream(),
                       reinterpret_cast<const bf16*>(q.data_ptr()), reinterpret_cast<const bf16*>(k.data_ptr()),
                       cosb.data_ptr<float>(), sinb.data_ptr<float>(), reinterpret_cast<bf16*>(qo.data_ptr()),
                       reinterpret_cast<bf16*>(ko.data_ptr()), S, Hq, Hk, D, q_rows, items, backward ? -1.f : 1.f);
    HIP_CHECK_KERNEL();
    return {qo, ko};
  }
  hipLaunchKernelGGL(rope_kernel, dim3((unsigned)grid), dim3(block), 0, stream.stream(),
                     reinterpret_cast<const bf16*>(q.data_ptr()),
                     reinterpret_cast<const bf16*>(k.data_ptr()),
                     cosb.data_ptr<float>(), sinb.data_ptr<float>(),
                     reinterpret_cast<bf16*>(qo.data_ptr()),
                     reinterpret_cast<bf16*>(ko.data_ptr()),
                     S, Hq, Hk, D, q_rows, total_rows, backward ? -1.f : 1.f);
  HIP_CHECK_KERNEL();
  return {qo, ko};
}

namespace {

// Rows of q, k and v side by side, and the three apart, q and k rotated as above (JOIN: back again, by the angles'
// negatives). Bound by reading and writing all of it once: 8192 rows of 32 + 2 x 8 heads of 128 32 us either way (6.3
// TB/s); three copies and the rotation took 73, that and a concatenation 89. A thread has 8 columns of a head and
// the 8 that are rotated with them.
template <bool JOIN>
__global__ __launch_bounds__(256) void rope_split_kernel(bf16* __restrict__ all, bf16* __restrict__ q, bf16* __restrict__ k,
                                                         bf16* __restrict__ v, const float* __restrict__ cosb,
                                                         const float* __restrict__ sinb, int S, int Hq, int Hk, int D,
                                                         long items) {
  const long id = (long)blockIdx.x * 256 + threadIdx.x;
  if (id >= items) return;
  const int chunks = D / 16, heads = Hq + 2 * Hk;
  const int c = (int)(id % chunks) * 8, h = (int)(id / chunks % heads);
  const long row = id / chunks / heads;
  bf16* const whole = all + (row * heads + h) * D + c;
  bf16* const apart = (h < Hq ? q + (row * Hq + h) * D : h < Hq + Hk ? k + (row * Hk + h - Hq) * D
                                                                     : v + (row * Hk + h - Hq - Hk) * D) + c;
  const bf16* from = JOIN ? apart : whole;
  bf16* to = JOIN ? whole : apart;
  bf16x8 x1 = *reinterpret_cast<const bf16x8*>(from), x2 = *reinterpret_cast<const bf16x8*>(from + D / 2);
  if (h < Hq + Hk) rotate8(x1, x2, cosb + row % S * D + c, sinb + row % S * D + c, JOIN ? -1.f : 1.f);
  *reinterpret_cast<bf16x8*>(to) = x1;
  *reinterpret_cast<bf16x8*>(to + D / 2) = x2;
}

template <bool JOIN>
void split(const at::Tensor& all, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& cosb,
           const at::Tensor& sinb) {
  const int B = q.size(0), S = q.size(1), Hq = q.size(2), Hk = k.size(2), D = q.size(3);
  for (const at::Tensor* t : {&all, &q, &k, &v})
    TORCH_CHECK(t->is_cuda() && t->device() == all.device() && t->scalar_type() == at::kBFloat16 && t->is_contiguous() &&
                    (uintptr_t)t->data_ptr() % 16 == 0, "rope_split: bf16, whole, at multiples of 16 bytes");
  for (const at::Tensor* t : {&cosb, &sinb})
    TORCH_CHECK(t->device() == all.device() && t->scalar_type() == at::kFloat && t->dim() == 2 && t->is_contiguous() &&
                    t->size(0) >= S && t->size(1) == D && (uintptr_t)t->data_ptr() % 16 == 0,
                "rope_split: cos, sin [S, D] f32");
  const std::vector<int64_t> kv{B, S, Hk, D};
  TORCH_CHECK(D >= 16 && D % 16 == 0 && k.sizes() == at::IntArrayRef(kv) && v.sizes() == at::IntArrayRef(kv) &&
                  all.numel() == (int64_t)B * S * (Hq + 2 * Hk) * D, "rope_split: shapes");
  const long items = (long)B * S * (Hq + 2 * Hk) * (D / 16);
  if (items == 0) return;
  TORCH_CHECK(items < 1l << 32, "rope_split: too many rows");
  auto at_ = [](const at::Tensor& t) { return reinterpret_cast<bf16*>(t.data_ptr()); };
  hipLaunchKernelGGL((rope_split_kernel<JOIN>), dim3((unsigned)((items + 255) / 256)), dim3(256), 0,
                     c10::hip::getCurrentHIPStream().stream(), at_(all), at_(q), at_(k), at_(v), cosb.data_ptr<float>(),
                     sinb.data_ptr<float>(), S, Hq, Hk, D, items);
  HIP_CHECK_KERNEL();
}

}  // namespace

// qkv [B, S, (Hq + 2 Hk) D] -> q [B, S, Hq, D] and k [B, S, Hk, D] rotated, v [B, S, Hk, D]
std::tuple<at::Tensor, at::Tensor, at::Tensor> rope_split(const at::Tensor& qkv, const at::Tensor& cosb,
                                                          const at::Tensor& sinb, int64_t Hq, int64_t Hk) {
  TORCH_CHECK(qkv.dim() == 3 && cosb.dim() == 2 && Hq >= 1 && Hk >= 1 && qkv.size(2) == (Hq + 2 * Hk) * cosb.size(1),
              "rope_split: qkv [B, S, (Hq + 2 Hk) D]");
  const int64_t B = qkv.size(0), S = qkv.size(1), D = cosb.size(1);
  auto q = at::empty({B, S, Hq, D}, qkv.options()), k = at::empty({B, S, Hk, D}, qkv.options()), v = at::empty_like(k);
  split<false>(qkv, q, k, v, cosb, sinb);
  return {q, k, v};
}

// its gradient: of the three -> of qkv
at::Tensor rope_join(const at::Tensor& dq, const at::Tensor& dk, const at::Tensor& dv, const at::Tensor& cosb,
                     const at::Tensor& sinb) {
  TORCH_CHECK(dq.dim() == 4 && dk.dim() == 4 && dv.dim() == 4, "rope_join: [B, S, H, D]");
  auto all = at::empty({dq.size(0), dq.size(1), (dq.size(2) + 2 * dk.size(2)) * dq.size(3)}, dq.options());
  split<true>(all, dq, dk, dv, cosb, sinb);
  return all;
}

// What a decode step begins with: rows of the embedding for its tokens, and rows of the rotary tables, as float32, for
// its positions. One launch: torch's two gathers, two casts and index_select are 12 us for one sequence of 4096 columns
// (of a step of 430) and 21 for 16, this 3. A block has 2048 columns of an embedding row, or 256 entries of both tables.
// Negative positions count from the end, as an index does; a token or position that is none gives NaN.
template <typename T>
__global__ __launch_bounds__(256) void token_rows_kernel(const long* __restrict__ ids, const bf16* __restrict__ table,
                                                         long vocab, int W, const long* __restrict__ pos,
                                                         const T* __restrict__ cosb, const T* __restrict__ sinb, long places,
                                                         int D, bf16* __restrict__ x, float* __restrict__ c,
                                                         float* __restrict__ s, int strips, int row_blocks, long entries) {
  if ((int)blockIdx.x < row_blocks) {
    const long row = blockIdx.x / strips, id = ids[row];
    const int col = (blockIdx.x % strips * 256 + threadIdx.x) * 8;
    if (col >= W) return;
    const unsigned nan = 0x7fc07fc0u;
    uint4 v{nan, nan, nan, nan};
    if (id >= 0 && id < vocab) v = *reinterpret_cast<const uint4*>(table + id * W + col);
    *reinterpret_cast<uint4*>(x + row * W + col) = v;
    return;
  }
  const long i = (long)(blockIdx.x - row_blocks) * 256 + threadIdx.x;
  if (i >= entries) return;
  long p = pos[i / D];
  if (p < 0) p += places;
  const bool in = p >= 0 && p < places;
  const long at = in ? p * D + i % D : 0;
  c[i] = in ? (float)cosb[at] : NAN;
  s[i] = in ? (float)sinb[at] : NAN;
}

// ids [..], table [vocab, W] bf16, pos [S], cos and sin [places, D] bf16 or float32
// -> {table[ids], cos[pos] and sin[pos] float32}
std::tuple<at::Tensor, at::Tensor, at::Tensor> token_rows(const at::Tensor& ids, const at::Tensor& table,
                                                          const at::Tensor& pos, const at::Tensor& cos,
                                                          const at::Tensor& sin) {
  for (const at::Tensor* t : {&ids, &table, &pos, &cos, &sin})
    TORCH_CHECK(t->is_cuda() && t->device() == ids.device() && t->is_contiguous(), "token_rows: whole tensors on one GPU");
  TORCH_CHECK(ids.scalar_type() == at::kLong && pos.scalar_type() == at::kLong && pos.dim() == 1 && table.dim() == 2 &&
                  table.scalar_type() == at::kBFloat16 && table.size(1) % 8 == 0 && (uintptr_t)table.data_ptr() % 16 == 0,
              "token_rows: 64-bit indices, table [vocab, W] bf16, W%8 == 0");
  TORCH_CHECK(cos.dim() == 2 && cos.size(0) > 0 && cos.sizes() == sin.sizes() && cos.scalar_type() == sin.scalar_type() &&
                  (cos.scalar_type() == at::kBFloat16 || cos.scalar_type() == at::kFloat),
              "token_rows: cos and sin [places, D], bf16 or float32");
  const c10::DeviceGuard guard(ids.device());
  auto shape = ids.sizes().vec();
  const long W = table.size(1), D = cos.size(1), S = pos.size(0), T = ids.numel();
  shape.push_back(W);
  auto x = at::empty(shape, table.options()), c = at::empty({S, D}, cos.options().dtype(at::kFloat)), s = at::empty_like(c);
  const long strips = (W + 2047) / 2048, row_blocks = T * strips, blocks = row_blocks + (S * D + 255) / 256;
  TORCH_CHECK(blocks < (1l << 24) && W < (1l << 31) && D < (1l << 31), "token_rows: too many rows");
  if (blocks == 0) return {x, c, s};
  const auto launch = [&](auto t) {
    using E = decltype(t);
    hipLaunchKernelGGL((token_rows_kernel<E>), dim3((unsigned)blocks), dim3(256), 0,
                       c10::hip::getCurrentHIPStream().stream(), ids.data_ptr<long>(),
                       reinterpret_cast<const bf16*>(table.data_ptr()), table.size(0), (int)W, pos.data_ptr<long>(),
                       reinterpret_cast<const E*>(cos.data_ptr()), reinterpret_cast<const E*>(sin.data_ptr()), cos.size(0),
                       (int)D, reinterpret_cast<bf16*>(x.data_ptr()), c.data_ptr<float>(), s.data_ptr<float>(), (int)strips,
                       (int)row_blocks, S * D);
  };
  if (cos.scalar_type() == at::kFloat) launch(float{});
  else launch(bf16{});
  HIP_CHECK_KERNEL();
  return {x, c, s};
}

}  // namespace amd_ops
