// Launches of y = x w^T by the tiles of gemm_tile.h (linear_grad.hip has the rest). The library's tiles of 256 x 256
// are as fast where they fill the chip's rounds and the sum is short, and leave CUs idle otherwise: here tiles and sums
// are cut as the gradients' are. us, library -> here, bf16 of unit variance, the weights not in a cache:
//   1001 x 14336 -> 4096 136 -> 113 (256 rows, 4 parts), 1001 x 21504 -> 4096 240 -> 155, 3003 x 2048 -> 2816 43 -> 37,
//   4096 x 4096 -> 6144 167 -> 161, 6001 x 4096 -> 4096 161 -> 151; 8192 x 4096 -> 6144 278 and 288, which stays the library's.
// The squared ReLU of a feed-forward layer's inner results is formed on the way out (6600 x 4096 -> 21504: a pass of 92 us
// less, of some 800). So is the gate's product with the other half of a gated one (linear_glu): the tiles' columns are 16
// of either weight in turn, and a lane has both sums. Against two products by the faster of library and kernel and a pass
// over both: 511 rows, 4096 -> 14336 137 -> 102 us, 2738 541 -> 461, 8192 1403 -> 1287, 14560 x 2048 -> 4096 457 -> 377; its
// error against 64 bits 0.0017, theirs 0.0031. ops/linear.py (output_own, squared_own, gated_own) has the rules and what they were
// fitted to.
#include <ATen/ATen.h>

#include "common.h"
#include "linear_tiles.h"

namespace amd_ops {
namespace lg {

void launch_out(const Args& a, unsigned blocks, hipStream_t stream) {
  const auto launch = [&](auto parts_, auto extra_, auto relu2_) {
    hipLaunchKernelGGL((linear_tile_kernel<Y, false, decltype(parts_)::value, decltype(extra_)::value, decltype(relu2_)::value>),
                       dim3(blocks), dim3(gt::THREADS), gt::SMEM, stream, a);
    HIP_CHECK_KERNEL();
  };
  using Yes = std::true_type;
  using No = std::false_type;
  if (a.parts > 1) a.rank ? launch(Yes{}, Yes{}, No{}) : launch(Yes{}, No{}, No{});
  else if (a.relu2) launch(No{}, No{}, Yes{});
  else a.rank ? launch(No{}, Yes{}, No{}) : launch(No{}, No{}, No{});
}

void launch_glu(const Args& a, unsigned blocks, hipStream_t stream) {
  hipLaunchKernelGGL((linear_tile_kernel<GLU, false, false>), dim3(blocks), dim3(gt::THREADS), gt::SMEM, stream, a);
  HIP_CHECK_KERNEL();
}

}  // namespace lg
}  // namespace amd_ops
