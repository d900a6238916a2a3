// Fully connected product with shared weights: the family of functions product / gradient of
// x1 / of x2 / of the weights, each differentiable in terms of the others, on csrc/fc_flex.hip and - from the measured crossings on -
// the kernels generated for the descriptor (codegen/fullyconnected.py).
#include "shared_map.h"
#include "tables.h"

namespace cueq_host {
namespace py = pybind11;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

struct Unit {  // a generated object's entry points (include/cueq_amd_generated.h)
  int (*fwd)(int64_t, const void*, const void*, int64_t, const void*, int64_t, void*, int64_t, void*) = nullptr;
  int (*dx1)(int64_t, const void*, const void*, int64_t, const void*, int64_t, void*, int64_t, void*) = nullptr;
  int (*dx2)(int64_t, const void*, const void*, int64_t, const void*, int64_t, const void*, int64_t, void*, int64_t, void*) = nullptr;
  int (*dx12)(int64_t, const void*, const void*, int64_t, const void*, int64_t, const void*, int64_t, void*, int64_t, void*, int64_t, float*, void*) = nullptr;
  int (*dw_blocks)(int64_t) = nullptr;
  int (*dw)(int64_t, const void*, int64_t, const void*, int64_t, const void*, int64_t, float*, int64_t, void*) = nullptr;
  int64_t fwd_from = 0, dx_from = 0, dw_from = 0;  // rows from which on they are the faster ones
};

constexpr int64_t kChunks = 64;  // row chunks of the weight gradient's tiled products

struct GradShape {  // the weight blocks of one extent: parts (path, component) of the tiled products, components per block
  int K, N, parts = 0;
  std::vector<int64_t> table, w0;
  int on_device = -1;
  std::vector<int32_t> first{0};
};

// 2-byte rows where the second operand has several channels: weights packed for each direction (cueq_fc_pack), weight gradient by
// groups of four channels
struct Packed {
  enum { kBlocks, kParts, kPacks, kCoef, kGrads };
  DeviceTables fwd, back;  // in this order (kGrads: back)
  int fwd_longest = 0, dx_longest = 0, grad_tiles = 0;  // grad_tiles == 0: the weight gradient takes the tables of the other types
  int64_t fwd_pieces = 0, dx_pieces = 0;
  bool any() const { return fwd_longest > 0; }
};

struct FcOp {
  int64_t width1 = 0, n2 = 0, width_out = 0, numel = 0;
  bool mul_ir = false, covers_in = true, covers_out = true;
  int epv_ok = 0, most = 1;
  enum { kBlocks, kParts, kCoef, kGrads };
  DeviceTables fwd, back;  // in this order (kGrads and the tiled products': back)
  std::string coef;
  int fwd_tiles = 0, dx_tiles = 0, grad_tiles = 0;
  SharedMap<Unit> units;  // by element type code
  std::vector<GradShape> shapes;
  Packed packed;
  int64_t h_width = 0;
  int factors = 0;
  int64_t tiled_dw_from[2] = {1 << 30, 1 << 30};  // rows, by element size (4, 2)
  bool float_factors = false;  // bfloat16 rows: the weight gradient's factors H stay float32 (half rows: always)

  bool takes(at::ScalarType t) const { return (t == at::kFloat && (epv_ok & 1)) || ((t == at::kBFloat16 || t == at::kHalf) && (epv_ok & 2)); }
};
using OpPtr = std::shared_ptr<FcOp>;

void launched(int status, const char* what) {
  if (status != 0) throw CueqError(std::string(what) + ": launch failed");
}

// the weights as the rows kernels read them: as they are, or packed
at::Tensor weights_for(FcOp& op, const at::Tensor& w, bool packed, bool gradient, int code, hipStream_t stream) {
  if (!packed) return w;
  DeviceTables& tables = gradient ? op.packed.back : op.packed.fwd;
  const int64_t pieces = gradient ? op.packed.dx_pieces : op.packed.fwd_pieces;
  at::Tensor out = at::empty({pieces * 8}, w.options());
  check(lib().cueq_fc_pack(code, w.data_ptr(), out.data_ptr(), tables.on(w.device(), Packed::kPacks), tables.count(Packed::kPacks, 48), pieces, stream),
        "cueq_fc_pack");
  return out;
}

// cueq_fc_flex's word on the rows and on the tables
int rows_layout(const FcOp& op, const DeviceTables& t) { return (op.mul_ir ? 1 : 0) + 2 * (t.count(FcOp::kParts, 56) / t.count(FcOp::kBlocks, 24)); }

at::Tensor product(FcOp& op, const at::Tensor& w_, const at::Tensor& x1_, const at::Tensor& x2_, at::ScalarType dtype) {
  const at::Device device = x1_.device();
  const c10::DeviceGuard guard(device);
  const at::Tensor w = rows_of(w_, dtype), x1 = rows_of(x1_, dtype), x2 = rows_of(x2_, dtype);
  const int64_t Z = x1.size(0);
  const auto options = at::TensorOptions().dtype(dtype).device(device);
  const int code = dtype_code(dtype);
  const std::optional<Unit> unit = op.units.find(code);
  // (a first call that is captured into a HIP graph: the generated kernels have no tables to upload)
  const Unit* u = unit && (Z >= unit->fwd_from || !op.fwd.at_hand(device)) ? &*unit : nullptr;
  at::Tensor out = op.covers_out || u ? at::empty({Z, op.width_out}, options) : at::zeros({Z, op.width_out}, options);
  if (Z == 0) return out;
  hipStream_t stream = stream_of(device.index());
  if (u) {
    launched(u->fwd(Z, w.data_ptr(), x1.data_ptr(), op.width1, x2.data_ptr(), op.n2, out.data_ptr(), op.width_out, stream), "fully connected product");
    return out;
  }
  const bool packed = op.packed.any() && dtype != at::kFloat;
  const at::Tensor ww = weights_for(op, w, packed, false, code, stream);
  DeviceTables& t = packed ? op.packed.fwd : op.fwd;
  check(lib().cueq_fc_flex(code, 0, rows_layout(op, t), packed ? op.packed.fwd_longest : 0, Z, x1.data_ptr(), op.width1, ww.data_ptr(), x2.data_ptr(), op.n2, nullptr, 0, out.data_ptr(), op.width_out,
                           t.on(device, FcOp::kBlocks), t.count(FcOp::kBlocks, 24), t.on(device, FcOp::kParts), t.on<float>(device, packed ? int(Packed::kCoef) : int(FcOp::kCoef)),
                           op.fwd_tiles, op.most, static_cast<int>(op.n2), nullptr, nullptr, stream),
        "cueq_fc_flex");
  return out;
}

struct Grads {
  at::Tensor w, x1, x2;
};
// the gradients asked for, in the types given (w: float32 sums rounded once)
Grads gradients(FcOp& op, const at::Tensor& w_, const at::Tensor& x1_, const at::Tensor& x2_, const at::Tensor& g_, at::ScalarType dtype, bool need_w, bool need_1,
                bool need_2, at::ScalarType w_dtype, at::IntArrayRef w_sizes) {
  const at::Device device = g_.device();
  const c10::DeviceGuard guard(device);
  const at::Tensor g = rows_of(g_, dtype);
  // (what a gradient does not read may be undefined)
  const at::Tensor w = w_.defined() ? rows_of(w_, dtype) : w_, x1 = x1_.defined() ? rows_of(x1_, dtype) : x1_, x2 = x2_.defined() ? rows_of(x2_, dtype) : x2_;
  const int64_t Z = g.size(0);
  const auto options = at::TensorOptions().dtype(dtype).device(device);
  Grads r;
  if (Z == 0) {
    if (need_w) r.w = at::zeros(w_sizes, options.dtype(w_dtype));
    if (need_1) r.x1 = at::empty({0, op.width1}, options);
    if (need_2) r.x2 = at::empty({0, op.n2}, options);
    return r;
  }
  const int code = dtype_code(dtype);
  hipStream_t stream = stream_of(device.index());
  const std::optional<Unit> unit = op.units.find(code);
  if (need_1 || need_2) {
    const Unit* u = unit && (Z >= unit->dx_from || !op.back.at_hand(device)) ? &*unit : nullptr;
    // (without x2 - the gradient of x2 alone does not use it - any values do: what they scale is not asked for)
    const at::Tensor second = x2.defined() ? x2 : at::zeros({Z, op.n2}, options);
    if (need_1) r.x1 = op.covers_in || u ? at::empty({Z, op.width1}, options) : at::zeros({Z, op.width1}, options);
    if (need_2) r.x2 = at::empty({Z, op.n2}, options);
    if (u) {
      int both = -2;
      if (need_1 && need_2) {  // one pass over the common products (-2: not for this object)
        at::Tensor part = new_tensor({Z, 2 * op.n2}, at::kFloat, device);
        both = u->dx12(Z, w.data_ptr(), g.data_ptr(), op.width_out, second.data_ptr(), op.n2, x1.data_ptr(), op.width1, r.x1.data_ptr(), op.width1, r.x2.data_ptr(),
                       op.n2, part.data_ptr<float>(), stream);
        if (both != -2) launched(both, "fully connected gradients");
      }
      if (both == -2) {
        if (need_1)
          launched(u->dx1(Z, w.data_ptr(), g.data_ptr(), op.width_out, second.data_ptr(), op.n2, r.x1.data_ptr(), op.width1, stream), "fully connected gradient");
        if (need_2)
          launched(u->dx2(Z, w.data_ptr(), x1.data_ptr(), op.width1, second.data_ptr(), op.n2, g.data_ptr(), op.width_out, r.x2.data_ptr(), op.n2, stream),
                   "fully connected gradient");
      }
    } else {
      at::Tensor part, dx1 = r.x1;
      if (need_2) part = new_tensor({op.dx_tiles, Z, op.n2}, at::kFloat, device);
      if (!dx1.defined()) dx1 = at::empty({Z, op.width1}, options);  // (the gradient of x2 comes from the same products)
      const bool packed = op.packed.any() && dtype != at::kFloat;
      const at::Tensor ww = weights_for(op, w, packed, true, code, stream);
      DeviceTables& t = packed ? op.packed.back : op.back;
      check(lib().cueq_fc_flex(code, 1, rows_layout(op, t), packed ? op.packed.dx_longest : 0, Z, g.data_ptr(), op.width_out, ww.data_ptr(), second.data_ptr(), op.n2, need_2 ? x1.data_ptr() : nullptr,
                               need_2 ? op.width1 : 0, dx1.data_ptr(), op.width1, t.on(device, FcOp::kBlocks), t.count(FcOp::kBlocks, 24),
                               t.on(device, FcOp::kParts), t.on<float>(device, packed ? int(Packed::kCoef) : int(FcOp::kCoef)), op.dx_tiles, op.most, static_cast<int>(op.n2),
                               need_2 ? part.data_ptr<float>() : nullptr, need_2 ? r.x2.data_ptr() : nullptr, stream),
            "cueq_fc_flex");
    }
  }
  if (need_w) {
    const at::ScalarType out_dtype = w_dtype == at::kDouble ? at::kFloat : w_dtype;
    const Unit* u = unit && (Z >= unit->dw_from || !op.back.at_hand(device)) ? &*unit : nullptr;
    // The factors H_i = sum_k s_ik g_k are operands of a product, rounded to its type.  In half they leave its range long before the
    // gradient does (65 504: a scaled loss), and bfloat16 calls that were float32 throughout would lose a rounding's worth: both
    // contract float copies of their rows.  (Generated kernels: a product's own, in its own type.)
    const at::ScalarType dw_dtype = !u && (dtype == at::kHalf || (dtype == at::kBFloat16 && op.float_factors)) ? at::kFloat : dtype;
    const at::Tensor a1 = x1.to(dw_dtype), a2 = x2.to(dw_dtype), ag = g.to(dw_dtype);
    const int dw_code = dtype_code(dw_dtype);
    at::Tensor gw = new_tensor(w_sizes, out_dtype, device);
    if (!u && Z >= op.tiled_dw_from[dw_dtype == at::kFloat ? 0 : 1]) {
      DeviceTables& t = op.back;
      at::Tensor H = at::empty({Z, op.h_width}, ag.options()), x1t = op.mul_ir ? at::empty({Z, op.width1}, ag.options()) : a1;
      check(lib().cueq_fc_factors(dw_code, op.mul_ir, Z, a1.data_ptr(), op.width1, a2.data_ptr(), op.n2, ag.data_ptr(), op.width_out, t.on(device, FcOp::kGrads),
                                  t.count(FcOp::kGrads, 72), t.on<float>(device, FcOp::kCoef), t.on(device, FcOp::kBlocks), t.count(FcOp::kBlocks, 24), op.factors, H.data_ptr(), op.h_width, op.mul_ir ? x1t.data_ptr() : nullptr, stream),
            "cueq_fc_factors");
      for (size_t i = 0; i < op.shapes.size(); ++i) {
        const GradShape& q = op.shapes[i];
        const int64_t per = int64_t(q.K) * q.N;
        at::Tensor part = new_tensor({q.parts * kChunks, per}, at::kFloat, device);
        check(lib().cueq_gemm_table(dw_code, CUEQ_F32, 1, 1, q.K, q.N, Z, x1t.data_ptr(), op.width1, H.data_ptr(), op.h_width, part.data_ptr(), q.N,
                                    t.on<int64_t>(device, q.on_device), q.parts, kChunks, per, 1.0, 0, stream),
              "cueq_gemm_table");
        check(lib().cueq_sum_runs(part.data_ptr<float>(), static_cast<int>(per), static_cast<int>(q.w0.size()), q.first.data(), q.w0.data(),
                                  dtype_code(out_dtype), gw.data_ptr(), stream),
              "cueq_sum_runs");
      }
      r.w = w_dtype == out_dtype ? gw : gw.to(w_dtype);
      return r;
    }
    const bool by_channels = op.packed.grad_tiles > 0 && dw_dtype != at::kFloat;
    const int grad_tiles = by_channels ? op.packed.grad_tiles : op.grad_tiles;
    const int64_t chunks = u ? u->dw_blocks(Z) : lib().cueq_fc_flex_dw_chunks(Z, grad_tiles, by_channels);
    at::Tensor part = new_tensor({chunks, op.numel}, at::kFloat, device);
    if (u) {
      launched(u->dw(Z, x1.data_ptr(), op.width1, x2.data_ptr(), op.n2, g.data_ptr(), op.width_out, part.data_ptr<float>(), op.numel, stream),
               "fully connected weight gradient");
    } else {
      DeviceTables& t = by_channels ? op.packed.back : op.back;
      const int table = by_channels ? int(Packed::kGrads) : int(FcOp::kGrads);
      check(lib().cueq_fc_flex_dw(dw_code, op.mul_ir, by_channels, Z, a1.data_ptr(), op.width1, a2.data_ptr(), op.n2, ag.data_ptr(), op.width_out, t.on(device, table),
                                  t.count(table, 72), t.on<float>(device, by_channels ? int(Packed::kCoef) : int(FcOp::kCoef)), grad_tiles, op.numel,
                                  part.data_ptr<float>(), stream),
            "cueq_fc_flex_dw");
    }
    const int32_t first[2] = {0, static_cast<int32_t>(chunks)};
    const int64_t w0 = 0;
    check(lib().cueq_sum_runs(part.data_ptr<float>(), static_cast<int>(op.numel), 1, first, &w0, dtype_code(out_dtype), gw.data_ptr(), stream), "cueq_sum_runs");
    r.w = w_dtype == out_dtype ? gw : gw.to(w_dtype);
  }
  return r;
}

struct Box : torch::CustomClassHolder {
  OpPtr op;
  at::ScalarType dtype, w_dtype;
  std::vector<int64_t> w_sizes;
  Box(OpPtr o, at::ScalarType d, at::ScalarType wd, at::IntArrayRef s) : op(std::move(o)), dtype(d), w_dtype(wd), w_sizes(s.vec()) {}
};
using BoxPtr = c10::intrusive_ptr<Box>;

at::Tensor forward(const OpPtr& op, const at::Tensor& w, const at::Tensor& x1, const at::Tensor& x2, at::ScalarType dtype);
at::Tensor gradient_1(const OpPtr& op, const at::Tensor& w, const at::Tensor& g, const at::Tensor& x2, at::ScalarType dtype);
at::Tensor gradient_2(const OpPtr& op, const at::Tensor& w, const at::Tensor& x1, const at::Tensor& g, at::ScalarType dtype);
at::Tensor gradient_w(const OpPtr& op, const at::Tensor& x1, const at::Tensor& x2, const at::Tensor& g, at::ScalarType dtype, at::ScalarType w_dtype,
                      at::IntArrayRef w_sizes);

at::Tensor as(const at::Tensor& t, const at::Tensor& like) { return t.to(like.scalar_type()); }

template <typename Derived>
struct Base : torch::autograd::Function<Derived> {
  static BoxPtr keep(AutogradContext* ctx, BoxPtr box, const variable_list& tensors) {
    ctx->save_for_backward(tensors);
    ctx->saved_data["b"] = c10::IValue::make_capsule(box);
    return box;
  }
  static BoxPtr box_of(AutogradContext* ctx) { return c10::static_intrusive_pointer_cast<Box>(ctx->saved_data["b"].toCapsule()); }
};

struct Product : Base<Product> {
  static at::Tensor forward(AutogradContext* ctx, BoxPtr box, const at::Tensor& w, const at::Tensor& x1, const at::Tensor& x2) {
    keep(ctx, box, {w, x1, x2});
    return product(*box->op, w, x1, x2, box->dtype);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list out(4);
    if (!grads[0].defined()) return out;
    const BoxPtr b = box_of(ctx);
    const auto t = ctx->get_saved_variables();
    const bool nw = ctx->needs_input_grad(0), n1 = ctx->needs_input_grad(1), n2 = ctx->needs_input_grad(2);
    if (!at::GradMode::is_enabled()) {  // a plain backward: the gradients in one call
      const Grads r = gradients(*b->op, t[0], t[1], t[2], grads[0], b->dtype, nw, n1, n2, t[0].scalar_type(), t[0].sizes());
      out[1] = r.w;
      out[2] = n1 ? as(r.x1, t[1]) : at::Tensor();
      out[3] = n2 ? as(r.x2, t[2]) : at::Tensor();
      return out;
    }
    if (nw) out[1] = gradient_w(b->op, t[1], t[2], grads[0], b->dtype, t[0].scalar_type(), t[0].sizes());
    if (n1) out[2] = as(gradient_1(b->op, t[0], grads[0], t[2], b->dtype), t[1]);
    if (n2) out[3] = as(gradient_2(b->op, t[0], t[1], grads[0], b->dtype), t[2]);
    return out;
  }
};

struct Gradient1 : Base<Gradient1> {
  static at::Tensor forward(AutogradContext* ctx, BoxPtr box, const at::Tensor& w, const at::Tensor& g, const at::Tensor& x2) {
    keep(ctx, box, {w, g, x2});
    return gradients(*box->op, w, at::Tensor(), x2, g, box->dtype, false, true, false, at::kFloat, {}).x1;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list out(4);
    if (!grads[0].defined()) return out;
    const BoxPtr b = box_of(ctx);
    const auto t = ctx->get_saved_variables();
    const at::Tensor& c = grads[0];
    if (ctx->needs_input_grad(0)) out[1] = gradient_w(b->op, c, t[2], t[1], b->dtype, t[0].scalar_type(), t[0].sizes());
    if (ctx->needs_input_grad(1)) out[2] = as(cueq_host::forward(b->op, t[0], c, t[2], b->dtype), t[1]);
    if (ctx->needs_input_grad(2)) out[3] = as(gradient_2(b->op, t[0], c, t[1], b->dtype), t[2]);
    return out;
  }
};

struct Gradient2 : Base<Gradient2> {
  static at::Tensor forward(AutogradContext* ctx, BoxPtr box, const at::Tensor& w, const at::Tensor& x1, const at::Tensor& g) {
    keep(ctx, box, {w, x1, g});
    return gradients(*box->op, w, x1, at::Tensor(), g, box->dtype, false, false, true, at::kFloat, {}).x2;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list out(4);
    if (!grads[0].defined()) return out;
    const BoxPtr b = box_of(ctx);
    const auto t = ctx->get_saved_variables();
    const at::Tensor& c = grads[0];
    if (ctx->needs_input_grad(0)) out[1] = gradient_w(b->op, t[1], c, t[2], b->dtype, t[0].scalar_type(), t[0].sizes());
    if (ctx->needs_input_grad(1)) out[2] = as(gradient_1(b->op, t[0], t[2], c, b->dtype), t[1]);
    if (ctx->needs_input_grad(2)) out[3] = as(cueq_host::forward(b->op, t[0], t[1], c, b->dtype), t[2]);
    return out;
  }
};

struct GradientW : Base<GradientW> {
  static at::Tensor forward(AutogradContext* ctx, BoxPtr box, const at::Tensor& x1, const at::Tensor& x2, const at::Tensor& g) {
    keep(ctx, box, {x1, x2, g});
    return gradients(*box->op, at::Tensor(), x1, x2, g, box->dtype, true, false, false, box->w_dtype, box->w_sizes).w;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list out(4);
    if (!grads[0].defined()) return out;
    const BoxPtr b = box_of(ctx);
    const auto t = ctx->get_saved_variables();
    const at::Tensor& c = grads[0];
    if (ctx->needs_input_grad(0)) out[1] = as(gradient_1(b->op, c, t[2], t[1], b->dtype), t[0]);
    if (ctx->needs_input_grad(1)) out[2] = as(gradient_2(b->op, c, t[0], t[2], b->dtype), t[1]);
    if (ctx->needs_input_grad(2)) out[3] = as(cueq_host::forward(b->op, c, t[0], t[1], b->dtype), t[2]);
    return out;
  }
};

at::Tensor forward(const OpPtr& op, const at::Tensor& w, const at::Tensor& x1, const at::Tensor& x2, at::ScalarType dtype) {
  if (!wants_graph({w, x1, x2})) return product(*op, w, x1, x2, dtype);
  return Product::apply(c10::make_intrusive<Box>(op, dtype, w.scalar_type(), w.sizes()), w, x1, x2);
}
at::Tensor gradient_1(const OpPtr& op, const at::Tensor& w, const at::Tensor& g, const at::Tensor& x2, at::ScalarType dtype) {
  if (!wants_graph({w, g, x2})) return gradients(*op, w, at::Tensor(), x2, g, dtype, false, true, false, at::kFloat, {}).x1;
  return Gradient1::apply(c10::make_intrusive<Box>(op, dtype, w.scalar_type(), w.sizes()), w, g, x2);
}
at::Tensor gradient_2(const OpPtr& op, const at::Tensor& w, const at::Tensor& x1, const at::Tensor& g, at::ScalarType dtype) {
  if (!wants_graph({w, x1, g})) return gradients(*op, w, x1, at::Tensor(), g, dtype, false, false, true, at::kFloat, {}).x2;
  return Gradient2::apply(c10::make_intrusive<Box>(op, dtype, w.scalar_type(), w.sizes()), w, x1, g);
}
at::Tensor gradient_w(const OpPtr& op, const at::Tensor& x1, const at::Tensor& x2, const at::Tensor& g, at::ScalarType dtype, at::ScalarType w_dtype,
                      at::IntArrayRef w_sizes) {
  if (!wants_graph({x1, x2, g})) return gradients(*op, at::Tensor(), x1, x2, g, dtype, true, false, false, w_dtype, w_sizes).w;
  return GradientW::apply(c10::make_intrusive<Box>(op, dtype, w_dtype, w_sizes), x1, x2, g);
}

// None unless it is a plain eager call of shapes and types the launches take
py::object direct(const OpPtr& op, const at::Tensor& w, const at::Tensor& x1, const at::Tensor& x2) {
  if (!ordinary(x1) || !ordinary(x2) || !ordinary(w) || !unwatched() || x1.dim() != 2 || x2.dim() != 2 || w.dim() != 2 || x1.size(1) != op->width1 ||
      x2.size(1) != op->n2 || x1.size(0) != x2.size(0) || w.size(0) != 1 || w.size(1) != op->numel || w.device() != x1.device() || x2.device() != x1.device() ||
      x1.scalar_type() != x2.scalar_type() || !op->takes(x1.scalar_type()) || dtype_code(w.scalar_type()) < 0)
    return py::none();
  return py::cast(forward(op, w, x1, x2, x1.scalar_type()));
}

}  // namespace

void bind_fully_connected(py::module_& m) {
  py::class_<FcOp, OpPtr>(m, "FcOp")
      .def(py::init([](int64_t width1, int64_t n2, int64_t width_out, int64_t numel, bool mul_ir, bool covers_in, bool covers_out, int epv_ok, int most,
                       const py::tuple& tables, const py::tuple& tiles) {
        auto op = std::make_shared<FcOp>();
        op->width1 = width1, op->n2 = n2, op->width_out = width_out, op->numel = numel;
        op->mul_ir = mul_ir, op->covers_in = covers_in, op->covers_out = covers_out, op->epv_ok = epv_ok, op->most = most;
        op->coef = tables[5].cast<std::string>();
        for (int t : {0, 1, 5}) op->fwd.add(tables[t].cast<std::string>());
        for (int t : {2, 3, 5, 4}) op->back.add(tables[t].cast<std::string>());
        op->fwd_tiles = tiles[0].cast<int>(), op->dx_tiles = tiles[1].cast<int>(), op->grad_tiles = tiles[2].cast<int>();
        return op;
      }))
      .def("add_unit", [](FcOp& op, int code, const std::vector<uintptr_t>& f, int64_t fwd_from, int64_t dx_from, int64_t dw_from) {
        Unit u;
        u.fwd = reinterpret_cast<decltype(u.fwd)>(f.at(0)), u.dx1 = reinterpret_cast<decltype(u.dx1)>(f.at(1)), u.dx2 = reinterpret_cast<decltype(u.dx2)>(f.at(2));
        u.dx12 = reinterpret_cast<decltype(u.dx12)>(f.at(3)), u.dw_blocks = reinterpret_cast<decltype(u.dw_blocks)>(f.at(4));
        u.dw = reinterpret_cast<decltype(u.dw)>(f.at(5));
        u.fwd_from = fwd_from, u.dx_from = dx_from, u.dw_from = dw_from;
        op.units.set(code, u);
      })
      // paths in the order of the weight-gradient table: (w0, a0, K, components, N, components of the result)
      .def("add_tiled_dw", [](FcOp& op, const py::list& paths, int64_t from4, int64_t from2) {
        op.tiled_dw_from[0] = from4;
        op.tiled_dw_from[1] = from2;
        int64_t h = 0;
        for (const auto& item : paths) {
          const py::tuple t = py::reinterpret_borrow<py::tuple>(item);
          const int64_t w0 = t[0].cast<int64_t>(), a0 = t[1].cast<int64_t>();
          const int K = t[2].cast<int>(), d = t[3].cast<int>(), N = t[4].cast<int>();
          GradShape* q = nullptr;
          for (auto& s : op.shapes)
            if (s.K == K && s.N == N) q = &s;
          if (!q) {
            op.shapes.emplace_back();
            q = &op.shapes.back();
            q->K = K, q->N = N;
          }
          for (int i = 0; i < d; ++i) {
            q->table.insert(q->table.end(), {a0 + int64_t(i) * K, h + int64_t(i) * N, int64_t(q->parts) * kChunks * K * N});
            ++q->parts;
          }
          q->w0.push_back(w0);
          q->first.push_back(static_cast<int32_t>(q->parts * kChunks));
          h += int64_t(d) * N;
          op.factors += d * t[5].cast<int>();
        }
        for (auto& q : op.shapes) q.on_device = op.back.add(q.table);
        op.h_width = h;
      })
      .def("add_packed", [](FcOp& op, const py::tuple& tables, const py::tuple& longest, const py::tuple& pieces, int grad_tiles) {
        auto& p = op.packed;
        for (int t : {0, 1, 4}) p.fwd.add(tables[t].cast<std::string>());
        for (int t : {2, 3, 5}) p.back.add(tables[t].cast<std::string>());
        p.fwd.add(op.coef), p.back.add(op.coef);
        p.back.add(tables[6].cast<std::string>());
        p.fwd_longest = longest[0].cast<int>(), p.dx_longest = longest[1].cast<int>(), p.grad_tiles = grad_tiles;
        p.fwd_pieces = pieces[0].cast<int64_t>(), p.dx_pieces = pieces[1].cast<int64_t>();
      })
      .def("keep_float_factors", [](FcOp& op) { op.float_factors = true; })
      .def("takes", [](const FcOp& op, const at::Tensor& x) { return op.takes(x.scalar_type()); })
      .def("direct", &direct)
      .def("forward", [](const OpPtr& op, const at::Tensor& w, const at::Tensor& x1, const at::Tensor& x2) { return forward(op, w, x1, x2, x1.scalar_type()); })
      .def("gradients", [](const OpPtr& op, const at::Tensor& w, const at::Tensor& x1, const at::Tensor& x2, const at::Tensor& g, bool nw, bool n1, bool n2) {
        const Grads r = gradients(*op, w, x1, x2, g, x1.scalar_type(), nw, n1, n2, w.scalar_type(), w.sizes());
        auto out = [](const at::Tensor& t) { return t.defined() ? py::cast(t) : py::object(py::none()); };
        return py::make_tuple(out(r.w), out(r.x1), out(r.x2));
      });
}

}  // namespace cueq_host
