// What the parts of the host module share: the entry points of the kernel library, loaded at run time, and small helpers
// around PyTorch's allocator and streams.
#pragma once

#include <ATen/hip/HIPContext.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <torch/extension.h>

#include <string>

#include "cueq_amd.h"

namespace cueq_host {

#define CUEQ_HOST_ENTRIES(X)                                                                                                     \
  X(cueq_last_error) X(cueq_set_option) X(cueq_u1d_plan_destroy) X(cueq_u1d_workspace_size) X(cueq_u1d_run)                      \
  X(cueq_segment_csr_workspace) X(cueq_segment_csr_build) X(cueq_segment_csr_build_async) X(cueq_trimul_bwd_parts)                \
  X(cueq_trimul_saved_bytes) X(cueq_trimul_workspace_bytes) X(cueq_trimul_fwd)                                         \
  X(cueq_linear_flex) X(cueq_linear_flex_dw_chunks) X(cueq_linear_flex_dw) X(cueq_sum_runs) X(cueq_linear_rows) X(cueq_linear_rows_mul_ir) \
  X(cueq_linear_dw_mul_ir_items) X(cueq_linear_dw_mul_ir) X(cueq_gemm_tn_items) X(cueq_gemm_tn) X(cueq_gemm_table) \
  X(cueq_fc_flex) X(cueq_fc_flex_dw_chunks) X(cueq_fc_flex_dw) X(cueq_fc_factors) X(cueq_fc_pack) X(cueq_rows_mean) X(cueq_normalize3)

// The library is the one the ctypes binding loaded (CUEQ_AMD_LIBRARY may name another build), so nothing is linked.
struct Library {
#define X(name) decltype(&::name) name = nullptr;
  CUEQ_HOST_ENTRIES(X)
#undef X
};
Library& lib();

struct CueqError : std::runtime_error {
  using std::runtime_error::runtime_error;
};
inline void check(int status, const char* what) {
  if (status != CUEQ_OK) throw CueqError(std::string(what) + " failed (status " + std::to_string(status) + "): " + lib().cueq_last_error());
}

// follows CUEQ_DETERMINISTIC / CUEQ_FORCE_GENERIC of the process's environment, at every uniform-1d launch (called with the GIL held)
void sync_options();

inline int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return CUEQ_F32;
    case at::kDouble: return CUEQ_F64;
    case at::kHalf: return CUEQ_F16;
    case at::kBFloat16: return CUEQ_BF16;
    default: return -1;
  }
}
inline hipStream_t stream_of(c10::DeviceIndex device) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device).stream(); }
inline at::Tensor new_tensor(at::IntArrayRef sizes, at::ScalarType dtype, at::Device device) {
  return at::empty(sizes, at::TensorOptions().dtype(dtype).device(device));
}

// An ordinary CUDA tensor whose data the kernels may read: not a tracer's, functorch's or a subclass's tensor.
inline bool ordinary(const at::Tensor& t) {
  static const c10::DispatchKeySet odd = c10::DispatchKeySet(
      {c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
       c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
  // (with a tangent of forward-mode differentiation it goes the way that refuses it: the launches here would drop the tangent)
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(odd) && !t._fw_grad(/*level=*/0).defined();
}
// nothing watches the calls (torch.jit.trace, dispatch modes): the direct path may be taken
bool unwatched();

bool wants_graph(const std::vector<at::Tensor>& tensors);  // gradients are recorded and some tensor asks for one

inline bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }  // a HIP graph

// (offsets[nrows + 1], perm[n]) grouping batch ids by output row; cached per index tensor in eager mode
std::pair<at::Tensor, at::Tensor> segment_csr(const at::Tensor& index, int64_t nrows);

void bind_uniform_1d(pybind11::module_& m);
void bind_triangle(pybind11::module_& m);
void bind_linear(pybind11::module_& m);
void bind_fully_connected(pybind11::module_& m);
void bind_rows(pybind11::module_& m);

}  // namespace cueq_host
