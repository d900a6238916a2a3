// Row-wise operations between the products of a layer.
#include "host.h"

namespace cueq_host {
namespace py = pybind11;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

// Sums over the batch rows grouped onto every row -> means (rows that collect none stay as they are).  Its own derivative: linear.
struct RowsMean : torch::autograd::Function<RowsMean> {
  static at::Tensor launch(const at::Tensor& x, const at::Tensor& offsets) {
    const c10::DeviceGuard guard(x.device());
    const at::Tensor in = x.contiguous();
    at::Tensor out = new_tensor(in.sizes(), in.scalar_type(), in.device());
    check(lib().cueq_rows_mean(dtype_code(in.scalar_type()), in.size(0), in.size(1), in.data_ptr(), offsets.data_ptr<int64_t>(), out.data_ptr(),
                               stream_of(in.device().index())),
          "cueq_rows_mean");
    return out;
  }
  static at::Tensor run(const at::Tensor& x, const at::Tensor& offsets) { return wants_graph({x}) ? apply(x, offsets) : launch(x, offsets); }

  static at::Tensor forward(AutogradContext* ctx, at::Tensor x, at::Tensor offsets) {
    ctx->save_for_backward({offsets});
    return launch(x, offsets);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    if (!grads[0].defined()) return {at::Tensor(), at::Tensor()};
    const at::Tensor offsets = ctx->get_saved_variables()[0];
    return {at::GradMode::is_enabled() ? run(grads[0], offsets) : launch(grads[0], offsets), at::Tensor()};
  }
};

// None for anything but a plain eager call (the caller then counts the degrees with PyTorch).  Under capture, and for index tensors
// without a version counter, the grouping is not kept and would have to be built again.
py::object rows_mean(const at::Tensor& sums, const at::Tensor& index) {
  if (!unwatched() || !ordinary(sums) || !ordinary(index) || sums.dim() != 2 || index.dim() != 1 || index.device() != sums.device() ||
      (index.scalar_type() != at::kInt && index.scalar_type() != at::kLong) || dtype_code(sums.scalar_type()) < 0 || index.is_inference() || !index.is_contiguous() ||
      sums.size(0) >= (int64_t(1) << 31) || capturing())
    return py::none();
  return py::cast(RowsMean::run(sums, segment_csr(index, sums.size(0)).first));
}

}  // namespace

void bind_rows(py::module_& m) { m.def("rows_mean", &rows_mean); }

}  // namespace cueq_host
