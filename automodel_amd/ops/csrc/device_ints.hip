// A few host integers as a device tensor, by way of a kernel's arguments. A copy from
// pageable memory waits until the stream has come to it: with one per decode step the host
// issued nothing while the GPU worked, and the GPU had nothing to do meanwhile (6 layer runs
// of 2048 columns, one sequence: 473 us a step, 403 now; 8 sequences of 4096 columns: 867
// and 823).

#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <climits>

#include "common.h"
#include "ops_api.h"

namespace amd_ops {

namespace {
constexpr int PER_LAUNCH = 960;        // of 4 KB of arguments
struct Ints {
  int v[PER_LAUNCH];
};
}  // namespace

__global__ __launch_bounds__(256) void device_ints_kernel(const Ints a, int* __restrict__ out, int n) {
  for (int i = threadIdx.x; i < n; i += 256) out[i] = a.v[i];
}

at::Tensor device_ints(at::IntArrayRef values, at::Device device) {
  TORCH_CHECK(device.is_cuda(), "device_ints: a GPU");
  const c10::DeviceGuard guard(device);
  const int64_t n = (int64_t)values.size();
  auto out = at::empty({n}, at::TensorOptions().dtype(at::kInt).device(device));
  for (int64_t i0 = 0; i0 < n; i0 += PER_LAUNCH) {
    const int part = (int)std::min<int64_t>(n - i0, PER_LAUNCH);
    Ints a;
    for (int i = 0; i < part; ++i) {
      TORCH_CHECK(values[i0 + i] >= INT_MIN && values[i0 + i] <= INT_MAX, "device_ints: int32");
      a.v[i] = (int)values[i0 + i];
    }
    for (int i = part; i < PER_LAUNCH; ++i) a.v[i] = 0;
    device_ints_kernel<<<dim3(1), dim3(256), 0, c10::hip::getCurrentHIPStream()>>>(
        a, out.data_ptr<int>() + i0, part);
    HIP_CHECK_KERNEL();
  }
  return out;
}

}  // namespace amd_ops
