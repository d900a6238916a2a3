// The uniform-1d operator: batch modes and row counts resolved once per call shape, launches and the backward without the
// interpreter.
#include "host.h"

#include <mutex>
#include <unordered_map>

namespace cueq_host {
namespace py = pybind11;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

enum { kAuto = -1, kShared = 0, kBatched = 1, kIndexed = 2 };

// A strong reference to the Python plan, given back with the interpreter's lock held.
struct PyHold {
  PyObject* object;
  explicit PyHold(PyObject* o) : object(o) {}
  PyHold(const PyHold&) = delete;
  ~PyHold() {
    if (!object || !Py_IsInitialized()) return;
    py::gil_scoped_acquire gil;
    Py_DECREF(object);
  }
};

struct Plan {
  int nin = 0, nout = 0;
  std::vector<int64_t> widths;
  std::vector<int> out_source;  // per output: the input whose element type it takes, -1: the arithmetic type
  at::ScalarType math = at::kFloat;
  PyObject* owner = nullptr;  // weak reference to the Python plan, which creates device plans and gradient plans
  std::vector<void*> handles;
  std::mutex mutex;

  ~Plan() {
    for (void* h : handles) lib().cueq_u1d_plan_destroy(static_cast<cueq_u1d_plan*>(h));
    if (owner && Py_IsInitialized()) {
      py::gil_scoped_acquire gil;
      Py_DECREF(owner);
    }
  }
  PyObject* python() const {  // (lock held) new reference
    PyObject* o = PyWeakref_GetObject(owner);
    TORCH_CHECK(o && o != Py_None, "uniform_1d: the plan is gone");
    Py_INCREF(o);
    return o;
  }
};

struct Key {
  std::vector<int64_t> v;
  bool operator==(const Key& o) const { return v == o.v; }
};
struct KeyHash {
  size_t operator()(const Key& k) const {
    uint64_t h = 1469598103934665603ull;
    for (int64_t x : k.v) h = (h ^ static_cast<uint64_t>(x)) * 1099511628211ull;
    return h;
  }
};

// One call shape of one plan: modes, rows and types of every buffer, and the argument array with all that does not change.
struct Record : c10::intrusive_ptr_target {
  std::shared_ptr<Plan> plan;
  std::vector<int> modes, index_of;
  std::vector<int64_t> rows;
  int64_t batch = 1;
  int nindex = 0;
  c10::DeviceIndex device = 0;
  cueq_u1d_plan* handle = nullptr;
  std::vector<at::ScalarType> types;  // of every buffer
  std::vector<cueq_u1d_buffer> buffers;
  std::mutex mutex;
  struct Backward {
    c10::intrusive_ptr<Record> record;
    uint64_t computed;
  };
  std::unordered_map<uint64_t, Backward> backward;  // by the inputs that ask for a gradient
};
using RecordPtr = c10::intrusive_ptr<Record>;

// (lock held) the record of a call shape: element types, device plan, kernels compiled where that is switched on
RecordPtr make_record(const std::shared_ptr<Plan>& plan, std::vector<int> modes, std::vector<int> index_of, std::vector<int64_t> rows, int64_t batch,
                      const std::vector<at::ScalarType>& in_types, const std::vector<at::ScalarType>& index_types, c10::DeviceIndex device) {
  auto r = c10::make_intrusive<Record>();
  const int n = plan->nin + plan->nout;
  r->plan = plan;
  r->modes = std::move(modes);
  r->index_of = std::move(index_of);
  r->rows = std::move(rows);
  r->batch = batch;
  r->nindex = static_cast<int>(index_types.size());
  r->device = device;
  r->buffers.resize(n);
  r->types = in_types;
  for (int o = 0; o < plan->nout; ++o) r->types.push_back(plan->out_source[o] < 0 ? plan->math : in_types[plan->out_source[o]]);
  for (int b = 0; b < n; ++b) {
    cueq_u1d_buffer& u = r->buffers[b];
    u = cueq_u1d_buffer{};
    u.rows = r->rows[b];
    u.dtype = dtype_code(r->types[b]);
    u.batch_dim = r->modes[b];
    if (r->modes[b] == kIndexed) u.index_is_64 = index_types[r->index_of[b]] == at::kLong ? 1 : 0;
  }
  py::object owner = py::reinterpret_steal<py::object>(plan->python());
  bool narrow = !in_types.empty() && c10::elementSize(in_types[0]) == 2;
  for (auto t : in_types) narrow = narrow && t == in_types[0];
  if (narrow) owner.attr("ensure_io")(py::cast(in_types[0]));
  r->handle = reinterpret_cast<cueq_u1d_plan*>(owner.attr("handle")(py::cast(at::Device(at::kCUDA, device))).cast<uintptr_t>());
  return r;
}

variable_list launch(const Record& r, const at::Tensor* inputs, const at::Tensor* indices) {
  const Plan& p = *r.plan;
  {
    py::gil_scoped_acquire gil;  // (a backward runs without it, and the program may be assigning to the environment)
    sync_options();
  }
  const at::Device device(at::kCUDA, r.device);
  const c10::DeviceGuard guard(device);
  c10::SmallVector<cueq_u1d_buffer, 12> bufs(r.buffers.begin(), r.buffers.end());
  c10::SmallVector<at::Tensor, 4> keep;
  for (int b = 0; b < p.nin; ++b) {
    const at::Tensor& t = inputs[b];
    if (t.is_contiguous()) {
      bufs[b].data = t.data_ptr();
    } else {
      keep.push_back(t.contiguous());
      bufs[b].data = keep.back().data_ptr();
    }
    if (r.modes[b] == kIndexed) bufs[b].index = indices[r.index_of[b]].data_ptr();
  }
  variable_list outs;
  outs.reserve(p.nout);
  for (int b = p.nin; b < p.nin + p.nout; ++b) {
    outs.push_back(new_tensor({r.rows[b], p.widths[b]}, r.types[b], device));
    bufs[b].data = outs.back().data_ptr();
    if (r.modes[b] == kIndexed) {
      const at::Tensor& idx = indices[r.index_of[b]];
      auto csr = segment_csr(idx, r.rows[b]);
      bufs[b].index = idx.data_ptr();
      bufs[b].csr_offsets = csr.first.data_ptr<int64_t>();
      bufs[b].csr_perm = csr.second.data_ptr<int64_t>();
      keep.push_back(std::move(csr.first));
      keep.push_back(std::move(csr.second));
    }
  }
  const int64_t bytes = lib().cueq_u1d_workspace_size(r.handle, bufs.data(), r.batch);
  at::Tensor ws;
  if (bytes > 0) ws = new_tensor({bytes}, at::kByte, device);
  check(lib().cueq_u1d_run(r.handle, bufs.data(), r.batch, bytes > 0 ? ws.data_ptr() : nullptr, bytes, stream_of(r.device)), "cueq_u1d_run");
  return outs;
}

struct ContextBox : torch::CustomClassHolder {
  RecordPtr record;
  std::shared_ptr<PyHold> owner;
};

struct Uniform1d : torch::autograd::Function<Uniform1d> {
  static variable_list run(const RecordPtr& r, const variable_list& tensors) {
    if (!wants_graph(tensors)) return launch(*r, tensors.data(), tensors.data() + r->plan->nin);
    auto box = c10::make_intrusive<ContextBox>();
    box->record = r;
    {
      py::gil_scoped_acquire gil;
      box->owner = std::make_shared<PyHold>(r->plan->python());
    }
    return apply(std::move(box), at::TensorList(tensors));
  }

  static variable_list forward(AutogradContext* ctx, c10::intrusive_ptr<ContextBox> box, at::TensorList tensors) {
    const Record& r = *box->record;
    ctx->save_for_backward(tensors.vec());
    auto outs = launch(r, tensors.data(), tensors.data() + r.plan->nin);
    ctx->saved_data["r"] = c10::IValue::make_capsule(std::move(box));
    return outs;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grad_outputs) {
    auto box = c10::static_intrusive_pointer_cast<ContextBox>(ctx->saved_data["r"].toCapsule());
    Record& r = *box->record;
    const Plan& p = *r.plan;
    variable_list tensors = ctx->get_saved_variables();
    variable_list result(1 + tensors.size());
    uint64_t needs = 0;
    for (int i = 0; i < p.nin; ++i)
      if (ctx->needs_input_grad(i)) needs |= 1ull << i;
    if (!needs) return result;
    // the grouping of a backward call: inputs, cotangents, indices
    variable_list args;
    args.reserve(tensors.size() + p.nout);
    args.insert(args.end(), tensors.begin(), tensors.begin() + p.nin);
    for (int o = 0; o < p.nout; ++o) {
      const int b = p.nin + o;
      at::Tensor g = grad_outputs[o];
      if (!g.defined()) g = at::zeros({r.rows[b], p.widths[b]}, at::TensorOptions().dtype(r.types[b]).device(at::Device(at::kCUDA, r.device)));
      if (g.scalar_type() != r.types[b]) g = g.to(r.types[b]);
      args.push_back(std::move(g));
    }
    args.insert(args.end(), tensors.begin() + p.nin, tensors.end());
    Record::Backward bw = gradient(r, needs);
    variable_list grads =
        at::GradMode::is_enabled() ? run(bw.record, args) : launch(*bw.record, args.data(), args.data() + p.nin + p.nout);
    int k = 0;
    for (int i = 0; i < p.nin; ++i) {
      if (!(bw.computed >> i & 1)) continue;
      if (needs >> i & 1) result[1 + i] = grads[k];
      ++k;
    }
    return result;
  }

  static Record::Backward gradient(Record& r, uint64_t needs) {
    {
      std::lock_guard<std::mutex> lock(r.mutex);
      auto hit = r.backward.find(needs);
      if (hit != r.backward.end()) return hit->second;
    }
    const Plan& p = *r.plan;
    Record::Backward bw;
    {
      py::gil_scoped_acquire gil;
      py::list flags;
      for (int i = 0; i < p.nin; ++i) flags.append(py::bool_(needs >> i & 1));
      py::object owner = py::reinterpret_steal<py::object>(p.python());
      py::tuple choice = owner.attr("backward_choice")(py::tuple(flags), py::cast(at::Device(at::kCUDA, r.device)));
      auto bplan = choice[0].attr("native").cast<std::shared_ptr<Plan>>();
      py::tuple computed = choice[1];
      std::vector<int> modes = r.modes, index_of = r.index_of;
      std::vector<int64_t> rows = r.rows;
      std::vector<at::ScalarType> index_types(r.nindex, at::kInt);
      for (int b = 0; b < p.nin + p.nout; ++b)
        if (r.modes[b] == kIndexed) index_types[r.index_of[b]] = r.buffers[b].index_is_64 ? at::kLong : at::kInt;
      bw.computed = 0;
      for (int i = 0; i < p.nin; ++i) {
        if (!computed[i].cast<bool>()) continue;
        bw.computed |= 1ull << i;
        modes.push_back(r.modes[i]);
        index_of.push_back(r.index_of[i]);
        rows.push_back(r.rows[i]);
      }
      bw.record = make_record(bplan, std::move(modes), std::move(index_of), std::move(rows), r.batch, r.types, index_types, r.device);
    }
    std::lock_guard<std::mutex> lock(r.mutex);
    return r.backward.emplace(needs, bw).first->second;
  }
};

// The operator of one descriptor: the plans of both arithmetic types behind one call.
struct Operator {
  std::shared_ptr<Plan> plan32, plan64;
  int fixed = -1;  // 0: always float32, 1: always float64, -1: the first input's type if it is one of the two, else float32
  std::unordered_map<Key, RecordPtr, KeyHash> records;

  // None for anything but a plain eager call with sound arguments (the Python path then runs it or says what is wrong)
  py::object call(const variable_list& inputs, const std::vector<std::optional<at::Tensor>>& in_index,
                  const std::vector<std::optional<at::Tensor>>& out_index, const std::vector<int64_t>& out_rows) {
    const auto outs = run(inputs, in_index, out_index, out_rows);
    if (outs.empty()) return py::none();
    return py::cast(outs);
  }

  // the three-operand products: weights, two operands (either may be gathered), one output (may be summed into rows)
  py::object product(const at::Tensor& w, const at::Tensor& x1, const at::Tensor& x2, const std::optional<at::Tensor>& i1, const std::optional<at::Tensor>& i2,
                     const std::optional<at::Tensor>& iout, const std::optional<int64_t>& size_out) {
    if (iout.has_value() != size_out.has_value()) return py::none();
    const auto outs = run({w, x1, x2}, {std::nullopt, i1, i2}, {iout}, {size_out.value_or(-1)});
    return outs.empty() ? py::none() : py::cast(outs[0]);
  }

  py::object indexed(const at::Tensor& w, const at::Tensor& x, const at::Tensor& index) {
    const auto outs = run({w.dim() > 2 ? w.flatten(1) : w, x}, {index, std::nullopt}, {std::nullopt}, {-1});
    return outs.empty() ? py::none() : py::cast(outs[0]);
  }

  variable_list run(const variable_list& inputs, const std::vector<std::optional<at::Tensor>>& in_index,
                    const std::vector<std::optional<at::Tensor>>& out_index, const std::vector<int64_t>& out_rows) {
    if (inputs.empty() || !unwatched()) return {};
    const at::ScalarType first = inputs[0].scalar_type();
    const bool f64 = fixed >= 0 ? fixed == 1 : first == at::kDouble;
    const std::shared_ptr<Plan>& plan = f64 ? plan64 : plan32;
    const Plan& p = *plan;
    if (static_cast<int>(inputs.size()) != p.nin || static_cast<int>(in_index.size()) != p.nin || static_cast<int>(out_index.size()) != p.nout) return {};
    const at::Device device = inputs[0].device();
    Key key;
    key.v.reserve(4 + 3 * p.nin + 2 * p.nout + 4);
    key.v.push_back(f64);
    key.v.push_back(device.index());
    variable_list args;
    args.reserve(p.nin + 4);
    for (int b = 0; b < p.nin; ++b) {
      const at::Tensor& t = inputs[b];
      if (!ordinary(t) || t.device() != device || t.dim() != 2 || t.size(1) != p.widths[b] || dtype_code(t.scalar_type()) < 0) return {};
      key.v.push_back(t.size(0));
      key.v.push_back(static_cast<int64_t>(t.scalar_type()));
      args.push_back(t);
    }
    variable_list indices;
    auto add_index = [&](const std::optional<at::Tensor>& idx) -> bool {
      if (!idx.has_value()) {
        key.v.push_back(-1);
        return true;
      }
      const at::Tensor& t = *idx;
      if (!ordinary(t) || t.device() != device || t.dim() != 1 || (t.scalar_type() != at::kInt && t.scalar_type() != at::kLong)) return false;
      key.v.push_back(2 * t.size(0) + (t.scalar_type() == at::kLong ? 1 : 0));
      indices.push_back(t.contiguous());
      return true;
    };
    for (const auto& i : in_index)
      if (!add_index(i)) return {};
    for (const auto& i : out_index)
      if (!add_index(i)) return {};
    for (int64_t r : out_rows) key.v.push_back(r);
    auto hit = records.find(key);
    RecordPtr rec;
    if (hit != records.end()) {
      rec = hit->second;
    } else {
      rec = resolve(plan, inputs, in_index, out_index, out_rows, indices, device.index());
      if (!rec) return {};
      if (records.size() >= 64) records.clear();  // (call shapes of a module are few; a stream of ever new batch sizes starts over)
      records.emplace(std::move(key), rec);
    }
    args.insert(args.end(), indices.begin(), indices.end());
    return Uniform1d::run(rec, args);
  }

  // the rules of uniform_1d.run_plan
  static RecordPtr resolve(const std::shared_ptr<Plan>& plan, const variable_list& inputs, const std::vector<std::optional<at::Tensor>>& in_index,
                           const std::vector<std::optional<at::Tensor>>& out_index, const std::vector<int64_t>& out_rows, const variable_list& indices,
                           c10::DeviceIndex device) {
    const Plan& p = *plan;
    const int n = p.nin + p.nout;
    std::vector<int> modes(n, kAuto), index_of(n, -1);
    std::vector<int64_t> rows(n, 0);
    int slot = 0;
    int64_t batch = kAuto;
    for (int b = 0; b < p.nin; ++b)
      if (in_index[b].has_value()) modes[b] = kIndexed, index_of[b] = slot++;
    for (int o = 0; o < p.nout; ++o) {
      const int64_t r = o < static_cast<int>(out_rows.size()) ? out_rows[o] : -1;
      if (out_index[o].has_value()) {
        if (r < 0) return {};
        modes[p.nin + o] = kIndexed, index_of[p.nin + o] = slot++;
        rows[p.nin + o] = r;
      } else if (r >= 0) {
        if (r == 1) {
          modes[p.nin + o] = kShared;
        } else {
          if (batch != kAuto && batch != r) return {};
          modes[p.nin + o] = kBatched;
          batch = r;
        }
      }
    }
    std::vector<int64_t> candidates;
    for (const auto& i : indices) candidates.push_back(i.size(0));
    for (int b = 0; b < p.nin; ++b)
      if (modes[b] != kIndexed && inputs[b].size(0) != 1) candidates.push_back(inputs[b].size(0));
    if (batch == kAuto) batch = candidates.empty() ? 1 : candidates[0];
    for (int64_t c : candidates)
      if (c != batch) return {};
    for (int b = 0; b < p.nin; ++b) {
      rows[b] = inputs[b].size(0);
      if (modes[b] == kAuto) modes[b] = rows[b] == 1 && batch != 1 ? kShared : kBatched;
    }
    for (int b = p.nin; b < n; ++b) {
      if (modes[b] == kIndexed) continue;
      if (modes[b] == kShared) rows[b] = 1;
      else modes[b] = kBatched, rows[b] = batch;
    }
    std::vector<at::ScalarType> types, index_types;
    for (const auto& t : inputs) types.push_back(t.scalar_type());
    for (const auto& i : indices) index_types.push_back(i.scalar_type());
    return make_record(plan, std::move(modes), std::move(index_of), std::move(rows), batch, types, index_types, device);
  }
};

}  // namespace

void bind_uniform_1d(py::module_& m) {
  py::class_<Plan, std::shared_ptr<Plan>>(m, "U1dPlan")
      .def(py::init([](int nin, int nout, std::vector<int64_t> widths, std::vector<int> out_source, bool f64, py::object owner) {
        auto p = std::make_shared<Plan>();
        p->nin = nin;
        p->nout = nout;
        p->widths = std::move(widths);
        p->out_source = std::move(out_source);
        p->math = f64 ? at::kDouble : at::kFloat;
        p->owner = PyWeakref_NewRef(owner.ptr(), nullptr);
        if (!p->owner) throw py::error_already_set();
        return p;
      }))
      .def("adopt", [](Plan& p, uintptr_t handle) { p.handles.push_back(reinterpret_cast<void*>(handle)); });
  // a resolved call: what run_plan keeps per call shape
  py::class_<Record, RecordPtr>(m, "U1dRecord")
      .def(py::init([](const std::shared_ptr<Plan>& plan, std::vector<int> modes, std::vector<int> index_of, std::vector<int64_t> rows, int64_t batch,
                       const std::vector<at::Tensor>& tensors) {
        std::vector<at::ScalarType> types, index_types;
        for (size_t i = 0; i < tensors.size(); ++i) (static_cast<int>(i) < plan->nin ? types : index_types).push_back(tensors[i].scalar_type());
        return make_record(plan, std::move(modes), std::move(index_of), std::move(rows), batch, types, index_types, tensors.at(0).device().index());
      }))
      .def("run", [](const RecordPtr& r, const variable_list& tensors) { return Uniform1d::run(r, tensors); });
  py::class_<Operator, std::shared_ptr<Operator>>(m, "U1dOperator")
      .def(py::init([](std::shared_ptr<Plan> plan32, std::shared_ptr<Plan> plan64, int fixed) {
        auto o = std::make_shared<Operator>();
        o->plan32 = std::move(plan32);
        o->plan64 = std::move(plan64);
        o->fixed = fixed;
        return o;
      }))
      .def("call", &Operator::call)
      .def("product", &Operator::product)
      .def("indexed", &Operator::indexed);
}

}  // namespace cueq_host
