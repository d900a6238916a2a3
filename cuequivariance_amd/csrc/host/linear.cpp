// Equivariant Linear with shared weights (uv,iu,iv): choice of the launches and the family of functions forward / input gradient /
// weight gradient, each differentiable in terms of the others.
#include "tables.h"

namespace cueq_host {
namespace py = pybind11;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {


struct RowsLaunch {  // cueq_linear_rows (d == 1 or ir_mul), cueq_linear_rows_mul_ir, or the tiled GEMM cueq_gemm_table (d == 0)
  int d, n, k, parts;
  double coeff;
  std::vector<int64_t> table;
  int on_device = -1;  // (d == 0) its number among the device tables
};
struct GradLaunch {  // one weight-gradient launch over strided components, or over mul_ir parts (table non-empty)
  int K, N;
  double coeff;
  int64_t a0, c0, da, dc;
  std::vector<int64_t> table;
  std::vector<int64_t> w_off;
  std::vector<int> components;  // per weight block
};

struct LinearOp {
  int64_t width_in = 0, width_out = 0, numel = 0;
  bool mul_ir = false, covers_in = true, covers_out = true;
  int epv_ok = 0;  // bit 0: float, bit 1: 2-byte elements
  enum { kBlocks, kParts, kGrads };
  DeviceTables fwd, back;  // the packed tables in this order (back: input gradient, then weight gradient), then those of tiled launches
  int fwd_tiles = 0, dx_tiles = 0, grad_tiles = 0;
  std::vector<RowsLaunch> fwd_rows[2], dx_rows[2];  // by element size (4, 2); empty: not for this shape
  std::vector<GradLaunch> grad_rows[2];
  int64_t rows_from[2] = {0, 0}, grad_rows_from[2] = {0, 0};  // from so many rows on the row-streaming launches are the faster ones

  bool takes(at::ScalarType t) const { return (t == at::kFloat && (epv_ok & 1)) || ((t == at::kBFloat16 || t == at::kHalf) && (epv_ok & 2)); }
};
using OpPtr = std::shared_ptr<LinearOp>;

// forward: x (Z, width_in) -> (Z, width_out); otherwise the input gradient, g (Z, width_out) -> (Z, width_in)
at::Tensor apply_rows(LinearOp& op, const at::Tensor& w_, const at::Tensor& x_, at::ScalarType dtype, bool forward) {
  const at::Device device = x_.device();
  const c10::DeviceGuard guard(device);
  const at::Tensor x = rows_of(x_, dtype), w = rows_of(w_, dtype);
  const int64_t Z = x.size(0), width = forward ? op.width_out : op.width_in, lda = forward ? op.width_in : op.width_out;
  const auto options = at::TensorOptions().dtype(dtype).device(device);
  at::Tensor out = (forward ? op.covers_out : op.covers_in) ? at::empty({Z, width}, options) : at::zeros({Z, width}, options);
  if (Z == 0) return out;
  const int e = dtype == at::kFloat ? 0 : 1, code = dtype_code(dtype);
  const auto& launches = forward ? op.fwd_rows[e] : op.dx_rows[e];
  hipStream_t stream = stream_of(device.index());
  DeviceTables& tables = forward ? op.fwd : op.back;
  // (a first call that is captured into a HIP graph: the launches whose tables are arguments, however few the rows)
  if (!launches.empty() && (Z >= op.rows_from[e] || !tables.at_hand(device))) {
    for (size_t i = 0; i < launches.size(); ++i) {
      const RowsLaunch& l = launches[i];
      if (l.d == 0)  // result columns n, contraction k; the weight block is contraction-major in the forward
        check(lib().cueq_gemm_table(code, code, 0, forward ? 1 : 0, Z, l.n, l.k, x.data_ptr(), lda, w.data_ptr(), forward ? l.n : l.k, out.data_ptr(), width,
                                    tables.on<int64_t>(device, l.on_device), l.parts, 1, 0, l.coeff, 0, stream),
              "cueq_gemm_table");
      else if (l.d == 1)
        check(lib().cueq_linear_rows(code, forward ? 1 : 0, Z, l.n, l.k, x.data_ptr(), lda, w.data_ptr(), op.numel, out.data_ptr(), width, l.table.data(), l.parts,
                                     l.coeff, stream),
              "cueq_linear_rows");
      else
        check(lib().cueq_linear_rows_mul_ir(code, forward ? 1 : 0, Z, l.n, l.k, x.data_ptr(), lda, w.data_ptr(), op.numel, out.data_ptr(), width,
                                            l.table.data(), l.parts, l.coeff, stream),
              "cueq_linear_rows_mul_ir");
    }
    return out;
  }
  check(lib().cueq_linear_flex(code, forward ? 0 : 1, Z, x.data_ptr(), lda, w.data_ptr(), out.data_ptr(), width, tables.on(device, LinearOp::kBlocks),
                               tables.count(LinearOp::kBlocks, 32), tables.on(device, LinearOp::kParts), forward ? op.fwd_tiles : op.dx_tiles, op.mul_ir ? 1 + 4 : 2 + 4, stream),
        "cueq_linear_flex");  // (2: rows in ir_mul, a block per component; 4: extents of 8 columns in any element type)
  return out;
}

at::Tensor weight_gradient(LinearOp& op, const at::Tensor& x_, const at::Tensor& g_, at::ScalarType w_dtype, at::IntArrayRef w_sizes) {
  const at::Device device = x_.device();
  const c10::DeviceGuard guard(device);
  const at::ScalarType dtype = x_.scalar_type();
  const at::Tensor x = rows_of(x_, dtype), g = rows_of(g_, dtype);
  const int64_t Z = x.size(0);
  if (Z == 0) return at::zeros(w_sizes, at::TensorOptions().dtype(w_dtype).device(device));
  const at::ScalarType out_dtype = w_dtype == at::kDouble ? at::kFloat : w_dtype;
  at::Tensor gw = new_tensor(w_sizes, out_dtype, device);
  const int e = dtype == at::kFloat ? 0 : 1, code = dtype_code(dtype), out_code = dtype_code(out_dtype);
  const int64_t es = dtype == at::kFloat ? 4 : 2;
  hipStream_t stream = stream_of(device.index());
  if (!op.grad_rows[e].empty() && (Z >= op.grad_rows_from[e] || !op.back.at_hand(device))) {
    for (const auto& l : op.grad_rows[e]) {
      const int n = static_cast<int>(l.w_off.size());
      std::vector<int32_t> first(n + 1, 0);
      at::Tensor part;
      if (!l.table.empty()) {
        const int64_t items = lib().cueq_linear_dw_mul_ir_items(Z, l.table.data(), n, first.data());
        part = new_tensor({items, int64_t(l.K) * l.N}, at::kFloat, device);
        check(lib().cueq_linear_dw_mul_ir(code, l.K, l.N, Z, x.data_ptr(), op.width_in, g.data_ptr(), op.width_out, l.table.data(), n, part.data_ptr<float>(),
                                          l.coeff, stream),
              "cueq_linear_dw_mul_ir");
      } else {
        int count = 0;
        for (int c : l.components) count += c;
        const int64_t items = lib().cueq_gemm_tn_items(Z, count), chunks = items / count;
        for (int b = 0; b < n; ++b) first[b + 1] = first[b] + static_cast<int32_t>(l.components[b] * chunks);
        part = new_tensor({items, int64_t(l.K) * l.N}, at::kFloat, device);
        check(lib().cueq_gemm_tn(code, l.K, l.N, Z, static_cast<char*>(x.data_ptr()) + l.a0 * es, op.width_in, l.da, static_cast<char*>(g.data_ptr()) + l.c0 * es,
                                 op.width_out, l.dc, count, part.data_ptr<float>(), l.coeff, stream),
              "cueq_gemm_tn");
      }
      check(lib().cueq_sum_runs(part.data_ptr<float>(), l.K * l.N, n, first.data(), l.w_off.data(), out_code, gw.data_ptr(), stream), "cueq_sum_runs");
    }
  } else {
    const int64_t chunks = lib().cueq_linear_flex_dw_chunks(Z, op.grad_tiles);
    at::Tensor part = new_tensor({chunks, op.numel}, at::kFloat, device);
    check(lib().cueq_linear_flex_dw(code, Z, x.data_ptr(), op.width_in, g.data_ptr(), op.width_out, op.back.on(device, LinearOp::kGrads), op.back.count(LinearOp::kGrads, 64),
                                    op.grad_tiles, op.numel, part.data_ptr<float>(), op.mul_ir, out_code, gw.data_ptr(), stream),
          "cueq_linear_flex_dw");
  }
  return w_dtype == out_dtype ? gw : gw.to(w_dtype);
}

struct Box : torch::CustomClassHolder {
  OpPtr op;
  at::ScalarType dtype;
  std::vector<int64_t> sizes;
  Box(OpPtr o, at::ScalarType d, at::IntArrayRef s) : op(std::move(o)), dtype(d), sizes(s.vec()) {}
};
using BoxPtr = c10::intrusive_ptr<Box>;
BoxPtr box_of(AutogradContext* ctx) { return c10::static_intrusive_pointer_cast<Box>(ctx->saved_data["b"].toCapsule()); }

at::Tensor forward(const OpPtr& op, const at::Tensor& w, const at::Tensor& x);
at::Tensor input_gradient(const OpPtr& op, const at::Tensor& g, const at::Tensor& w, at::ScalarType x_dtype);
at::Tensor weights_gradient(const OpPtr& op, const at::Tensor& x, const at::Tensor& g, at::ScalarType w_dtype, at::IntArrayRef w_sizes);

struct Forward : torch::autograd::Function<Forward> {
  static at::Tensor forward(AutogradContext* ctx, BoxPtr box, const at::Tensor& w, const at::Tensor& x) {
    ctx->save_for_backward({w, x});
    at::Tensor out = apply_rows(*box->op, w, x, x.scalar_type(), true);
    ctx->saved_data["b"] = c10::IValue::make_capsule(std::move(box));
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto t = ctx->get_saved_variables();
    const OpPtr op = box_of(ctx)->op;
    variable_list out(3);
    if (!grads[0].defined()) return out;
    if (ctx->needs_input_grad(1)) out[2] = input_gradient(op, grads[0], t[0], t[1].scalar_type());
    if (ctx->needs_input_grad(0)) out[1] = weights_gradient(op, t[1], grads[0], t[0].scalar_type(), t[0].sizes());
    return out;
  }
};

struct InputGradient : torch::autograd::Function<InputGradient> {  // dx = g W^T
  static at::Tensor forward(AutogradContext* ctx, BoxPtr box, const at::Tensor& g, const at::Tensor& w) {
    ctx->save_for_backward({g, w});
    at::Tensor out = apply_rows(*box->op, w, g, box->dtype, false);
    ctx->saved_data["b"] = c10::IValue::make_capsule(std::move(box));
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto t = ctx->get_saved_variables();
    const OpPtr op = box_of(ctx)->op;
    variable_list out(3);
    if (!grads[0].defined()) return out;
    if (ctx->needs_input_grad(0)) out[1] = cueq_host::forward(op, t[1], grads[0]).to(t[0].scalar_type());
    if (ctx->needs_input_grad(1)) out[2] = weights_gradient(op, grads[0], t[0], t[1].scalar_type(), t[1].sizes());
    return out;
  }
};

struct WeightGradient : torch::autograd::Function<WeightGradient> {  // dW = x^T g
  static at::Tensor forward(AutogradContext* ctx, BoxPtr box, const at::Tensor& x, const at::Tensor& g) {
    ctx->save_for_backward({x, g});
    at::Tensor out = weight_gradient(*box->op, x, g, box->dtype, box->sizes);
    ctx->saved_data["b"] = c10::IValue::make_capsule(std::move(box));
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto t = ctx->get_saved_variables();
    const OpPtr op = box_of(ctx)->op;
    variable_list out(3);
    if (!grads[0].defined()) return out;
    if (ctx->needs_input_grad(0)) out[1] = input_gradient(op, t[1], grads[0], t[0].scalar_type());
    if (ctx->needs_input_grad(1)) out[2] = cueq_host::forward(op, grads[0], t[0]).to(t[1].scalar_type());
    return out;
  }
};

at::Tensor forward(const OpPtr& op, const at::Tensor& w, const at::Tensor& x) {
  if (!wants_graph({w, x})) return apply_rows(*op, w, x, x.scalar_type(), true);
  return Forward::apply(c10::make_intrusive<Box>(op, x.scalar_type(), w.sizes()), w, x);
}
at::Tensor input_gradient(const OpPtr& op, const at::Tensor& g, const at::Tensor& w, at::ScalarType x_dtype) {
  if (!wants_graph({g, w})) return apply_rows(*op, w, g, x_dtype, false);
  return InputGradient::apply(c10::make_intrusive<Box>(op, x_dtype, at::IntArrayRef()), g, w);
}
at::Tensor weights_gradient(const OpPtr& op, const at::Tensor& x, const at::Tensor& g, at::ScalarType w_dtype, at::IntArrayRef w_sizes) {
  if (!wants_graph({x, g})) return weight_gradient(*op, x, g, w_dtype, w_sizes);
  return WeightGradient::apply(c10::make_intrusive<Box>(op, w_dtype, w_sizes), x, g);
}

// None unless it is a plain eager call of a shape and type the launches take
py::object direct(const OpPtr& op, const at::Tensor& w, const at::Tensor& x) {
  if (!ordinary(x) || !ordinary(w) || !unwatched() || x.dim() != 2 || x.size(1) != op->width_in || w.dim() != 2 || w.size(0) != 1 || w.size(1) != op->numel ||
      w.device() != x.device() || !op->takes(x.scalar_type()) || dtype_code(w.scalar_type()) < 0)
    return py::none();
  return py::cast(forward(op, w, x));
}

std::vector<RowsLaunch> rows_launches(const py::list& l, DeviceTables& tables) {
  std::vector<RowsLaunch> out;
  for (const auto& item : l) {
    const py::tuple t = py::reinterpret_borrow<py::tuple>(item);
    out.push_back({t[0].cast<int>(), t[1].cast<int>(), t[2].cast<int>(), t[4].cast<int>(), t[5].cast<double>(), t[3].cast<std::vector<int64_t>>()});
    if (out.back().d == 0) out.back().on_device = tables.add(out.back().table);
  }
  return out;
}

}  // namespace

void bind_linear(py::module_& m) {
  py::class_<LinearOp, OpPtr>(m, "LinearOp")
      .def(py::init([](int64_t width_in, int64_t width_out, int64_t numel, bool mul_ir, bool covers_in, bool covers_out, int epv_ok, const py::tuple& tables,
                       const py::tuple& tiles) {
        auto op = std::make_shared<LinearOp>();
        op->width_in = width_in, op->width_out = width_out, op->numel = numel;
        op->mul_ir = mul_ir, op->covers_in = covers_in, op->covers_out = covers_out, op->epv_ok = epv_ok;
        for (int t = 0; t < 5; ++t) (t < 2 ? op->fwd : op->back).add(tables[t].cast<std::string>());
        op->fwd_tiles = tiles[0].cast<int>(), op->dx_tiles = tiles[1].cast<int>(), op->grad_tiles = tiles[2].cast<int>();
        return op;
      }))
      // launches for many rows, elements of `es` bytes: lists of (d, columns, contraction, table, parts, coefficient)
      .def("add_rows", [](LinearOp& op, int es, int64_t from, const py::list& fwd, const py::list& dx) {
        const int e = es == 4 ? 0 : 1;
        op.fwd_rows[e] = rows_launches(fwd, op.fwd);
        op.dx_rows[e] = rows_launches(dx, op.back);
        op.rows_from[e] = from;
      })
      // lists of (K, N, coefficient, a0, c0, da, dc, table, weight offsets, components per weight block)
      .def("add_grads", [](LinearOp& op, int es, int64_t from, const py::list& launches) {
        const int e = es == 4 ? 0 : 1;
        op.grad_rows_from[e] = from;
        op.grad_rows[e].clear();
        for (const auto& item : launches) {
          const py::tuple t = py::reinterpret_borrow<py::tuple>(item);
          op.grad_rows[e].push_back({t[0].cast<int>(), t[1].cast<int>(), t[2].cast<double>(), t[3].cast<int64_t>(), t[4].cast<int64_t>(), t[5].cast<int64_t>(),
                                     t[6].cast<int64_t>(), t[7].cast<std::vector<int64_t>>(), t[8].cast<std::vector<int64_t>>(), t[9].cast<std::vector<int>>()});
        }
      })
      .def("takes", [](const LinearOp& op, const at::Tensor& x) { return op.takes(x.scalar_type()); })
      .def("direct", &direct)
      .def("forward", &forward)
      .def("dx", [](const OpPtr& op, const at::Tensor& w, const at::Tensor& g, const at::Tensor& x) { return apply_rows(*op, w, g, x.scalar_type(), false); })
      .def("dw", [](const OpPtr& op, const at::Tensor& x, const at::Tensor& g, const at::Tensor& w) {
        return weight_gradient(*op, x, g, w.scalar_type(), w.sizes());
      });
}

}  // namespace cueq_host
