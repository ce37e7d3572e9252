// Shared pieces of the native host path: from torch tensors to the C ABI of include/mi355q.h without Python.
//
// Why it exists: the kernels of a decode step take 3 .. 15 us each, and a Python wrapper of the same work
// (attribute look-ups, views, the dispatcher calling back into Python, a ctypes call of twenty arguments)
// took 20 .. 26 us per operator on an EPYC core, so the GPU waited for the host.  Here an operator
// costs its allocation and its launch.
#pragma once

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <cstdint>

#include "../../../include/mi355q.h"

namespace mi355q_host {

using at::Tensor;

inline int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kHalf: return MI355Q_F16;
    case at::kBFloat16: return MI355Q_BF16;
    case at::kFloat: return MI355Q_F32;
    default: return -1;
  }
}
inline bool is_16bit(at::ScalarType t) { return t == at::kHalf || t == at::kBFloat16; }

inline int require_dtype(at::ScalarType t) {
  const int c = dtype_code(t);
  TORCH_CHECK_TYPE(c >= 0, "unsupported dtype ", t);
  return c;
}

inline void check(int rc, const char* what) {
  TORCH_CHECK(rc == 0, "mi355q ", what, " failed (code ", rc, "): ", mi355q_last_error());
}

// the tensor's device for the time of a call (nothing to do where it is the current one already)
struct OnDevice {
  int before, dev;
  explicit OnDevice(const Tensor& t) : before(c10::hip::current_device()), dev(t.get_device()) {
    if (before != dev) c10::hip::set_device(static_cast<c10::DeviceIndex>(dev));
  }
  ~OnDevice() {
    if (before != dev) c10::hip::set_device(static_cast<c10::DeviceIndex>(before));
  }
  void* stream() const { return c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream(); }
};

inline Tensor empty(at::IntArrayRef sizes, at::ScalarType t, const Tensor& like) {
  return Tensor(at::detail::empty_cuda(sizes, t, like.device(), std::nullopt));
}

inline void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// Scratch of the current stream of `like`'s device with at least `bytes` bytes: the buffer that
// vllm_gcu_amd.kernels._runtime.workspace keeps per (device, stream).  Called with the GIL held; the buffers
// seen here are held, so a buffer that Python replaces by a larger one stays valid.
struct Scratch {
  char* p;
  size_t bytes;
};
Scratch workspace(const Tensor& like, void* stream, size_t bytes);

// memory ranges that hold weights in the kslab order
bool is_kslab(const Tensor& w);

void register_activation_ops();     // the operators without a weight: norm, activation, quantisation, routing, sum

}  // namespace mi355q_host
