// Native host path of ppo_amd: the extension module ppo_amd._native.
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include "scale.hpp"

namespace {

void* current_stream(const at::Device& device) {
  return c10::hip::getCurrentHIPStream(device.index()).stream();
}

// dst[k] = src[k] * scale (a one-element fp32 tensor) in one launch; all
// contiguous fp32 on one device.  Returns the library's status code.
int scale_grads(const std::vector<at::Tensor>& src, const std::vector<at::Tensor>& dst,
                const at::Tensor& scale) {
  TORCH_CHECK(!src.empty() && src.size() == dst.size() && src.size() <= ppo::kMaxScaleArrays,
              "scale_grads takes 1 to ", ppo::kMaxScaleArrays, " tensors");
  ppo::ScaleArray a[ppo::kMaxScaleArrays];
  for (size_t k = 0; k < src.size(); ++k) {
    TORCH_CHECK(src[k].scalar_type() == at::kFloat && dst[k].scalar_type() == at::kFloat &&
                    src[k].is_contiguous() && dst[k].is_contiguous() &&
                    src[k].numel() == dst[k].numel() && src[k].device() == scale.device() &&
                    dst[k].device() == scale.device(),
                "scale_grads takes contiguous fp32 tensors of one size on one device");
    a[k] = {src[k].const_data_ptr<float>(), dst[k].data_ptr<float>(), src[k].numel()};
  }
  TORCH_CHECK(scale.is_cuda() && scale.scalar_type() == at::kFloat && scale.numel() == 1,
              "scale must be a one-element fp32 GPU tensor");
  return ppo::launch_scale(a, (int)src.size(), scale.const_data_ptr<float>(),
                           current_stream(scale.device()));
}

}  // namespace

PYBIND11_MODULE(_native, m) {
  m.def("scale_grads", &scale_grads);
}
