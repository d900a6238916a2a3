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

constexpr double kNormalizeEps = 1e-12;  // of torch.nn.functional.normalize

void normalize3(int stage, const at::Tensor& x, const at::Tensor& g, const at::Tensor& v, at::Tensor& out, at::Tensor& out_x) {
  const c10::DeviceGuard guard(x.device());
  const auto data = [](const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; };
  check(lib().cueq_normalize3(dtype_code(x.scalar_type()), stage, x.size(0), data(x), data(g), data(v), kNormalizeEps, data(out), data(out_x),
                              stream_of(x.device().index())),
        "cueq_normalize3");
}

// x / max(|x|, eps) for rows of three, its gradient, and the gradient of that.  Beyond, PyTorch differentiates the formulas.
struct NormalizeGrad : torch::autograd::Function<NormalizeGrad> {
  static at::Tensor launch(const at::Tensor& g, const at::Tensor& x) {
    const at::Tensor xc = x.contiguous(), gc = g.contiguous();
    at::Tensor out = new_tensor(xc.sizes(), xc.scalar_type(), xc.device()), none;
    normalize3(1, xc, gc, none, out, none);
    return out;
  }
  static at::Tensor run(const at::Tensor& g, const at::Tensor& x) { return wants_graph({g, x}) ? apply(g, x) : launch(g, x); }

  static at::Tensor forward(AutogradContext* ctx, at::Tensor g, at::Tensor x) {
    ctx->save_for_backward({g, x});
    return launch(g, x);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const at::Tensor v = grads[0];
    if (!v.defined()) return {at::Tensor(), at::Tensor()};
    const auto saved = ctx->get_saved_variables();
    const at::Tensor &g = saved[0], &x = saved[1];
    const bool want_g = ctx->needs_input_grad(0), want_x = ctx->needs_input_grad(1);
    at::Tensor dg, dx;
    if (at::GradMode::is_enabled()) {
      if (want_g) dg = run(v, x);
      if (want_x) {
        const at::Tensor length = at::linalg_vector_norm(x, 2, {1}, true), through = length.lt(kNormalizeEps).logical_not();  // (a NaN stays one)
        const at::Tensor n = length.clamp_min(kNormalizeEps), y = x / n;
        const at::Tensor yv = (y * v).sum(1, true), yg = (y * g).sum(1, true), vg = (v * g).sum(1, true);
        dx = at::where(through, ((3 * yv * yg - vg) * y - yg * v - yv * g) / n / n, at::zeros({}, x.options()));
      }
      return {dg, dx};
    }
    const at::Tensor xc = x.contiguous(), gc = g.contiguous(), vc = v.contiguous();
    if (want_g) dg = new_tensor(xc.sizes(), xc.scalar_type(), xc.device());
    if (want_x) dx = new_tensor(xc.sizes(), xc.scalar_type(), xc.device());
    if (want_g || want_x) normalize3(2, xc, gc, vc, dg, dx);
    return {dg, dx};
  }
};

struct Normalize : torch::autograd::Function<Normalize> {
  static at::Tensor launch(const at::Tensor& x) {
    const at::Tensor xc = x.contiguous();
    at::Tensor out = new_tensor(xc.sizes(), xc.scalar_type(), xc.device()), none;
    normalize3(0, xc, none, none, out, none);
    return out;
  }
  static at::Tensor forward(AutogradContext* ctx, at::Tensor x) {
    ctx->save_for_backward({x});
    return launch(x);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    if (!grads[0].defined()) return {at::Tensor()};
    const at::Tensor x = ctx->get_saved_variables()[0];
    return {at::GradMode::is_enabled() ? NormalizeGrad::run(grads[0], x) : NormalizeGrad::launch(grads[0], x)};
  }
};

// None for anything but a plain eager call on float32 or float64 rows of three
py::object normalize(const at::Tensor& x) {
  if (!unwatched() || !ordinary(x) || x.dim() != 2 || x.size(1) != 3 || (x.scalar_type() != at::kFloat && x.scalar_type() != at::kDouble)) return py::none();
  return py::cast(wants_graph({x}) ? Normalize::apply(x) : Normalize::launch(x));
}

}  // namespace

void bind_rows(py::module_& m) {
  m.def("rows_mean", &rows_mean);
  m.def("normalize", &normalize);
}

}  // namespace cueq_host
