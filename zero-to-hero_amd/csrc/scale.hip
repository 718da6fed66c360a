// The losses' backward (loss.backward(), rl/deep/agents/ppo.py:169): the
// gradients the fused loss kernels wrote, times the incoming gradient of the
// total loss, in one launch.
#include <algorithm>

#include "common.hpp"
#include "scale.hpp"

namespace ppo {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));

// Scaled in place by exactly 1 -- loss.backward() on the loss itself -- nothing
// is read or written but the scalar: the forward kernel already wrote these
// gradients.
//
// What bounds it: HBM when it scales (8 bytes per element), the launch when it
// does not.  Measured on MI355X, forward + backward of the categorical loss (B =
// 8,388,608, A = 18, vf_clip): 488 us with a torch multiplication per gradient,
// 214 us of them those, 272 us with this launch finding a scale of 1.
struct ScaleTable {
  ScaleArray a[kMaxScaleArrays];
  int narr;
  int in_place;
};

// Workgroups: enough to fill the chip eight times over with 256 threads, few
// enough that a launch that finds the scale to be 1 ends in about 2 us.
constexpr long kScaleBlocks = 2048;

__global__ void __launch_bounds__(kBlock) scale_kernel(ScaleTable t,
                                                       const float* __restrict__ scale) {
  const float g = *scale;
  if (t.in_place && g == 1.0f) return;
  const long stride = (long)gridDim.x * blockDim.x;
  const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  for (int k = 0; k < t.narr; ++k) {
    const float* in = t.a[k].src;
    float* out = t.a[k].dst;
    const long n = t.a[k].numel;
    long tail = 0;
    if (((uintptr_t)in | (uintptr_t)out) % 16 == 0) {
      const long n4 = n / 4;
      for (long i = gid; i < n4; i += stride) {
        f4 x = __builtin_nontemporal_load(reinterpret_cast<const f4*>(in) + i);
        x[0] *= g;
        x[1] *= g;
        x[2] *= g;
        x[3] *= g;
        __builtin_nontemporal_store(x, reinterpret_cast<f4*>(out) + i);
      }
      tail = 4 * n4;
    }
    for (long i = tail + gid; i < n; i += stride) out[i] = in[i] * g;
  }
}

}  // namespace

int launch_scale(const ScaleArray* arrays, int narrays, const float* scale, void* stream) {
  if (narrays < 1 || narrays > kMaxScaleArrays || !scale) return PPO_ERR_INVALID_ARG;
  ScaleTable t = {};
  t.narr = narrays;
  t.in_place = 1;
  long most = 0;
  for (int k = 0; k < narrays; ++k) {
    t.a[k] = arrays[k];
    t.in_place = t.in_place && arrays[k].src == arrays[k].dst;
    most = std::max(most, (long)arrays[k].numel);
  }
  if (most == 0) return PPO_OK;
  const long blocks = std::min((most + 4L * kBlock - 1) / (4L * kBlock), kScaleBlocks);
  hipLaunchKernelGGL(scale_kernel, dim3((unsigned)blocks), dim3(kBlock), 0,
                     reinterpret_cast<hipStream_t>(stream), t, scale);
  return last_launch_status();
}

}  // namespace ppo
