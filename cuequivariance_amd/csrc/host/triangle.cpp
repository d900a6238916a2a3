// The triangle multiplicative update: argument checks, buffers and the backward without the interpreter around
// cueq_trimul_fwd / cueq_trimul_bwd.
#include "host.h"

namespace cueq_host {
namespace py = pybind11;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

constexpr int kWeights = 12;  // norm_in w, b, p_in w, b, g_in w, b, norm_out w, b, p_out w, b, g_out w, b

struct Call {
  int32_t code;
  int64_t B, N, D, Do;
  at::Device device;
  const void* w[kWeights];
  explicit Call(const at::Tensor& x, at::TensorList weights)
      : code(dtype_code(x.scalar_type())), B(x.size(0)), N(x.size(1)), D(x.size(3)), Do(weights[8].size(0)), device(x.device()) {
    for (int i = 0; i < kWeights; ++i) w[i] = weights[i].defined() ? weights[i].data_ptr() : nullptr;
  }
};

at::Tensor aligned(const at::Tensor& t) { return t.defined() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 ? t.clone() : t; }
variable_list aligned(at::TensorList ts) {
  variable_list out;
  for (const auto& t : ts) out.push_back(aligned(t));
  return out;
}
void* pointer(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// x (B, N, N, D), mask (B, N, N) or undefined, weights as above (undefined where absent), all contiguous in x's type; saved_bytes: a
// size of what is kept for the backward that the caller has promised (a traced graph), 0: as much as is needed
std::pair<at::Tensor, at::Tensor> trimul_fwd(const at::Tensor& x_, const at::Tensor& mask, at::TensorList weights, bool outgoing, double eps, int64_t saved_bytes = 0) {
  const at::Tensor x = aligned(x_);
  const variable_list w = aligned(weights);
  const Call c(x, w);
  const c10::DeviceGuard guard(c.device);
  at::Tensor out = new_tensor({c.B, c.N, c.N, c.Do}, x.scalar_type(), c.device);
  const int64_t needed = lib().cueq_trimul_saved_bytes(c.code, c.B, c.N, c.D, c.Do);
  TORCH_CHECK(!saved_bytes || saved_bytes >= needed, "triangle update: ", saved_bytes, " bytes promised for the backward, ", needed, " needed");
  at::Tensor saved = new_tensor({saved_bytes ? saved_bytes : needed}, at::kByte, c.device), ws;
  const int64_t bytes = lib().cueq_trimul_workspace_bytes(c.code, c.B, c.N, c.D, c.Do, 0, 0);
  if (bytes > 0) ws = new_tensor({bytes}, at::kByte, c.device);
  check(lib().cueq_trimul_fwd(c.code, c.B, c.N, c.D, c.Do, outgoing, eps, x.data_ptr(), pointer(mask), c.w, out.data_ptr(), saved.data_ptr(), pointer(ws), bytes,
                              stream_of(c.device.index())),
        "cueq_trimul_fwd");
  return {out, saved};
}

// [dx, the twelve weight gradients] for the bits of `need` (bit 0: x, bit 1 + i: weight i)
variable_list trimul_bwd(const at::Tensor& x_, const at::Tensor& mask, at::TensorList weights, const at::Tensor& saved, bool outgoing, uint32_t need,
                         const at::Tensor& dout_) {
  const at::Tensor x = aligned(x_);
  const variable_list w = aligned(weights);
  const Call c(x, w);
  const c10::DeviceGuard guard(c.device);
  uint32_t bits = need >> 1;
  for (int i = 0; i < kWeights; ++i)
    if (!weights[i].defined()) bits &= ~(1u << i);
  at::Tensor dx = new_tensor(x.sizes(), x.scalar_type(), c.device);
  variable_list out(1 + kWeights);
  void* grads[kWeights] = {};
  for (int i = 0; i < kWeights; ++i) {
    if (!(bits >> i & 1)) continue;
    out[1 + i] = new_tensor(weights[i].sizes(), x.scalar_type(), c.device);
    grads[i] = out[1 + i].data_ptr();
    if (x.numel() == 0) out[1 + i].zero_();
  }
  if (x.numel() != 0) {
    const at::Tensor dout = aligned(dout_.to(x.scalar_type()).contiguous());
    const int64_t bytes = lib().cueq_trimul_workspace_bytes(c.code, c.B, c.N, c.D, c.Do, 1, bits != 0);
    at::Tensor ws = new_tensor({bytes}, at::kByte, c.device);
    check(lib().cueq_trimul_bwd_parts(c.code, c.B, c.N, c.D, c.Do, outgoing, x.data_ptr(), pointer(mask), c.w, saved.data_ptr(), dout.data_ptr(), dx.data_ptr(),
                                      bits, grads, ws.data_ptr(), bytes, stream_of(c.device.index())),
          "cueq_trimul_bwd_parts");
  }
  if (need & 1) out[0] = dx;
  return out;
}

// (autograd takes defined tensors only: `present` says which of x, mask and the weights are there)
struct TriMul : torch::autograd::Function<TriMul> {
  static variable_list all(at::TensorList given, int64_t present) {
    variable_list t(2 + kWeights);
    size_t k = 0;
    for (int i = 0; i < 2 + kWeights; ++i)
      if (present >> i & 1) t[i] = given[k++];
    return t;
  }
  static at::Tensor forward(AutogradContext* ctx, bool outgoing, double eps, int64_t present, at::TensorList given) {
    const variable_list t = all(given, present);
    auto [out, saved] = trimul_fwd(t[0], t[1], at::TensorList(t).slice(2), outgoing, eps);
    variable_list keep = given.vec();
    keep.push_back(saved);
    ctx->save_for_backward(keep);
    ctx->saved_data["o"] = outgoing;
    ctx->saved_data["p"] = present;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const variable_list kept = ctx->get_saved_variables();
    const int64_t present = ctx->saved_data["p"].toInt();
    const variable_list t = all(kept, present);
    // (by what requires a gradient, not by what this call asks for: the traced operator only knows the former, and which
    // kernels run - hence the last bits of dx - must not depend on who asks)
    uint32_t need = 0;
    for (int i = 0; i < 2 + kWeights; ++i)
      if (i != 1 && t[i].defined() && t[i].requires_grad()) need |= i == 0 ? 1u : 1u << (i - 1);
    const auto got = trimul_bwd(t[0], t[1], at::TensorList(t).slice(2), kept.back(), ctx->saved_data["o"].toBool(), need, g[0]);
    variable_list out(3);
    for (int i = 0; i < 2 + kWeights; ++i)
      if (present >> i & 1) out.push_back(i == 0 ? got[0] : i == 1 ? at::Tensor() : got[i - 1]);
    return out;
  }
};

at::Tensor run(const at::Tensor& x, const std::optional<at::Tensor>& mask, const std::vector<std::optional<at::Tensor>>& weights, bool outgoing, double eps) {
  variable_list t{x, mask.value_or(at::Tensor())};
  for (const auto& w : weights) t.push_back(w.value_or(at::Tensor()));
  if (wants_graph(t)) {
    variable_list given;
    int64_t present = 0;
    for (size_t i = 0; i < t.size(); ++i)
      if (t[i].defined()) given.push_back(t[i]), present |= int64_t(1) << i;
    return TriMul::apply(outgoing, eps, present, at::TensorList(given));
  }
  return trimul_fwd(t[0], t[1], at::TensorList(t).slice(2), outgoing, eps).first;
}

// None unless everything is as the kernels take it: x (B, N, N, D), tensors contiguous, one element type, projections given
py::object direct(const at::Tensor& x, const std::optional<at::Tensor>& mask, const std::vector<std::optional<at::Tensor>>& weights, bool outgoing, double eps) {
  if (!ordinary(x) || x.dim() != 4 || !x.is_contiguous() || x.size(1) != x.size(2) || x.size(3) % 32 || !unwatched() || weights.size() != kWeights) return py::none();
  const at::ScalarType T = x.scalar_type();
  if (T != at::kFloat && T != at::kBFloat16 && T != at::kHalf) return py::none();
  const int64_t D = x.size(3);
  auto fits = [&](const std::optional<at::Tensor>& t, at::IntArrayRef sizes) {
    return !t.has_value() || (ordinary(*t) && t->scalar_type() == T && t->device() == x.device() && t->is_contiguous() && t->sizes() == sizes);
  };
  if (!fits(mask, {x.size(0), x.size(1), x.size(2)})) return py::none();
  for (int i : {2, 4, 8, 10})
    if (!weights[i].has_value() || weights[i]->dim() != 2) return py::none();
  const int64_t Do = weights[8]->size(0);
  const std::vector<int64_t> sizes[kWeights] = {{D}, {D}, {2 * D, D}, {2 * D}, {2 * D, D}, {2 * D}, {D}, {D}, {Do, D}, {Do}, {Do, D}, {Do}};
  for (int i = 0; i < kWeights; ++i)
    if (!fits(weights[i], sizes[i])) return py::none();
  return py::cast(run(x, mask, weights, outgoing, eps));
}

variable_list given(const std::vector<std::optional<at::Tensor>>& weights) {
  variable_list w;
  for (const auto& t : weights) w.push_back(t.value_or(at::Tensor()));
  return w;
}

}  // namespace

void bind_triangle(py::module_& m) {
  using OptionalList = std::vector<std::optional<at::Tensor>>;
  m.def("trimul", &run);
  m.def("trimul_direct", &direct);
  m.def("trimul_fwd", [](const at::Tensor& x, const std::optional<at::Tensor>& mask, const OptionalList& weights, bool outgoing, double eps, int64_t saved_bytes) {
    return trimul_fwd(x, mask.value_or(at::Tensor()), given(weights), outgoing, eps, saved_bytes);
  });
  m.def("trimul_bwd", [](const at::Tensor& x, const std::optional<at::Tensor>& mask, const OptionalList& weights, const at::Tensor& saved, bool outgoing,
                         uint32_t need, const at::Tensor& dout) {
    py::list out;
    for (const auto& t : trimul_bwd(x, mask.value_or(at::Tensor()), given(weights), saved, outgoing, need, dout)) out.append(t.defined() ? py::cast(t) : py::none());
    return out;
  });
}

}  // namespace cueq_host
