// csrc/native_device.h with host memory for the device: the calls of native_calls.cpp up to the launch, on a machine
// without a GPU.
#pragma once

#include <ATen/EmptyTensor.h>

namespace {

bool on_device(const at::Tensor& t) { return t.is_cpu(); }

at::Tensor empty_like_device(at::IntArrayRef sizes, const at::Tensor& like) {
  TORCH_CHECK_WITH(OutOfMemoryError, like.scalar_type() == at::kHalf, "host memory is out of bfloat16");
  return at::Tensor(at::detail::empty_cpu(sizes, like.scalar_type()));
}

void* current_stream() { return nullptr; }

}  // namespace
