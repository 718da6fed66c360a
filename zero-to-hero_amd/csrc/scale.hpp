// Scaling of saved gradients by a device scalar (scale.hip), for native.cpp.
#pragma once

#include <stdint.h>

namespace ppo {

constexpr int kMaxScaleArrays = 4;

struct ScaleArray {
  const float* src;
  float* dst;  // may equal src
  int64_t numel;
};

// dst[i] = src[i] * *scale for every array, in one launch on `stream`; where
// every dst is its src and the scale is 1, nothing is written.
int launch_scale(const ScaleArray* arrays, int narrays, const float* scale, void* stream);

}  // namespace ppo
