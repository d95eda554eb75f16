// The part of the framework's host path that runs on every call, in C++: argument checks,
// output allocation through PyTorch's caching allocator and the call into the kernel library
// (include/megalodon_hip.h).  Built by g++ against the installed PyTorch; no kernels here.
#pragma once

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/utils/pybind.h>

#include <optional>
#include <stdexcept>
#include <string>

#include "../../../include/megalodon_hip.h"

namespace mega_host {

namespace py = pybind11;
using at::Tensor;

// errors surface as RuntimeError, as everywhere in the package
[[noreturn]] inline void fail(const std::string& what) { throw std::runtime_error(what); }
inline void require(bool ok, const char* what) {
  if (!ok) fail(what);
}
inline void check(int code, const char* name) {
  if (code != MEGA_OK)
    fail(std::string(name) + " failed (code " + std::to_string(code) + "): " + mega_last_error());
}

inline void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// element type code of the C interface, -1 for a type it does not have
inline int code_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return MEGA_F32;
    case at::kBFloat16: return MEGA_BF16;
    case at::kHalf: return MEGA_F16;
    default: return -1;
  }
}

// what a tensor says is in its memory: a lazily conjugated or negated view keeps the sign in a bit that neither
// contiguous() nor data_ptr() looks at
inline bool lazy(const Tensor& t) { return t.is_conj() || t.is_neg(); }
inline Tensor stored(const Tensor& t) { return lazy(t) ? t.resolve_conj().resolve_neg() : t; }

// whether a forward-mode derivative travels with the tensor
inline bool has_tangent(const Tensor& t) { return t._fw_grad(/*level=*/0).defined(); }

void bind_decode(py::module_& m);
void bind_ops(py::module_& m);

}  // namespace mega_host
