// What native_calls.cpp needs to know of the device: which tensors lie on it, where results come from, which stream is
// current.
#pragma once

#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPStream.h>

namespace {

bool on_device(const at::Tensor& t) { return t.is_cuda(); }

at::Tensor empty_like_device(at::IntArrayRef sizes, const at::Tensor& like) {
  return at::Tensor(at::detail::empty_cuda(sizes, like.scalar_type(), like.device(), std::nullopt));
}

void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

}  // namespace
