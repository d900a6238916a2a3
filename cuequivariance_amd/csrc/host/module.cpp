// The host side of the hot launch paths in native code.  A forward and backward of a small batch costs a few launches; resolving
// the call, allocating the results and entering the backward in Python took several times as long (and the backward, which
// PyTorch runs on a thread of its own, had to wait for the interpreter): the step of 622 edges, 50 us of kernels, took 176 us.
// Everything here falls back to the Python path (by returning None) for calls that are not plain eager ones.
#include "host.h"

#include <dlfcn.h>

#include <cstdlib>
#include <list>
#include <mutex>

#include <torch/csrc/jit/frontend/tracer.h>

namespace cueq_host {

Library& lib() {
  static Library l;
  return l;
}

namespace {
PyObject* g_error_class = nullptr;

struct EnvOption {
  const char *env, *option;
  std::string seen;
  bool set = false;
} g_env[] = {{"CUEQ_DETERMINISTIC", "deterministic"}, {"CUEQ_FORCE_GENERIC", "force_generic"}};

void load(const std::string& path, pybind11::object error_class) {
  void* handle = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  if (!handle) throw std::runtime_error(std::string("cannot load ") + path + ": " + dlerror());
#define X(name)                                                                  \
  lib().name = reinterpret_cast<decltype(&::name)>(dlsym(handle, #name));        \
  if (!lib().name) throw std::runtime_error(path + " has no entry point " #name);
  CUEQ_HOST_ENTRIES(X)
#undef X
  g_error_class = error_class.release().ptr();
  for (auto& o : g_env) {  // (the library has read the environment itself when it was loaded)
    const char* v = std::getenv(o.env);
    o.set = v != nullptr;
    o.seen = v ? v : "";
  }
}

struct CsrEntry {
  at::Tensor index, offsets, perm;
  uint32_t version;
  int64_t nrows;
};
std::mutex g_csr_mutex;
std::list<CsrEntry> g_csr;  // most recently used first
}  // namespace

void sync_options() {
  for (auto& o : g_env) {
    const char* v = std::getenv(o.env);
    if ((v != nullptr) == o.set && (!v || o.seen == v)) continue;
    o.set = v != nullptr;
    o.seen = v ? v : "";
    lib().cueq_set_option(o.option, v && v[0] == '1' ? 1 : 0);
  }
}

bool unwatched() { return !torch::jit::tracer::isTracing() && !c10::impl::TorchDispatchModeTLS::any_modes_set(); }

bool wants_graph(const std::vector<at::Tensor>& tensors) {
  for (const auto& t : tensors)  // (a call without a graph would drop the tangent)
    TORCH_CHECK_NOT_IMPLEMENTED(!t.defined() || !t._fw_grad(/*level=*/0).defined(), "cuequivariance_amd: forward-mode differentiation is not implemented");
  if (!at::GradMode::is_enabled()) return false;
  for (const auto& t : tensors)
    if (t.defined() && t.requires_grad()) return true;
  return false;
}

namespace {
PyObject* key(const char* name) { return PyUnicode_InternFromString(name); }

PyObject* dict_of(PyObject* object) {  // borrowed: the attributes of an instance
  PyObject** d = _PyObject_GetDictPtr(object);
  return d ? *d : nullptr;
}
bool empty(PyObject* dict, PyObject* name) {  // there and without an entry
  PyObject* hooks = PyDict_GetItem(dict, name);
  return hooks && PyDict_Check(hooks) && PyDict_Size(hooks) == 0;
}

// The children of a module are of the classes it was built with, and a call of one runs its `forward` and nothing else.
bool untouched(PyObject* module, PyObject* built) {
  static PyObject* const modules = key("_modules");
  static PyObject* const hooks[] = {key("_forward_hooks"), key("_forward_pre_hooks"), key("_backward_hooks"), key("_backward_pre_hooks")};
  static PyObject* const replaced[] = {key("forward"), key("_compiled_call_impl")};
  PyObject* own = dict_of(module);
  PyObject* children = own ? PyDict_GetItem(own, modules) : nullptr;
  if (!children || !PyDict_Check(children)) return false;
  PyObject *name, *child;
  Py_ssize_t at = 0;
  while (PyDict_Next(children, &at, &name, &child)) {
    if (child == Py_None) continue;
    if (PySet_Contains(built, reinterpret_cast<PyObject*>(Py_TYPE(child))) != 1) return false;
    PyObject* d = dict_of(child);
    if (!d) return false;
    for (PyObject* h : hooks)
      if (!empty(d, h)) return false;
    for (PyObject* r : replaced)
      if (PyDict_Contains(d, r)) return false;
  }
  return true;
}

// The executor of class `kind` that a call of `module`'s child `name` (of class `outer`) ends in, None unless it may be run without those
// calls: nothing replaced, wrapped or hooked on the way, no hook on all modules.
pybind11::object executor(const pybind11::object& module, const pybind11::str& name, const pybind11::type& outer, const pybind11::type& kind,
                          const pybind11::object& built) {
  static PyObject* const global[] = {key("_global_backward_pre_hooks"), key("_global_backward_hooks"),        key("_global_forward_pre_hooks"),
                                     key("_global_forward_hooks"),      key("_global_forward_hooks_always_called"), key("_global_forward_hooks_with_kwargs")};
  static PyObject* const torch_module = PyModule_GetDict(PyImport_ImportModule("torch.nn.modules.module"));
  static PyObject *const modules = key("_modules"), *const inner = key("m");
  for (PyObject* g : global)
    if (!empty(torch_module, g)) return pybind11::none();
  if (!untouched(module.ptr(), built.ptr())) return pybind11::none();
  PyObject* f = PyDict_GetItem(PyDict_GetItem(dict_of(module.ptr()), modules), name.ptr());
  if (!f || reinterpret_cast<PyObject*>(Py_TYPE(f)) != outer.ptr() || !untouched(f, built.ptr())) return pybind11::none();
  PyObject* m = PyDict_GetItem(PyDict_GetItem(dict_of(f), modules), inner);
  if (!m || reinterpret_cast<PyObject*>(Py_TYPE(m)) != kind.ptr() || !untouched(m, built.ptr())) return pybind11::none();
  return pybind11::reinterpret_borrow<pybind11::object>(m);
}
}  // namespace

// Eager mode: built once per index tensor and cached (the build checks on the host that the ids are in range and skips the sort when
// they are sorted already).  While the current stream is being captured into a HIP graph the grouping is recorded into the graph
// instead (device-side work only, nothing cached), so every replay regroups from whatever the index buffer holds then.  Index
// tensors made under torch.inference_mode() carry no version counter and are not cached either.
std::pair<at::Tensor, at::Tensor> segment_csr(const at::Tensor& index, int64_t nrows) {
  const bool recorded = capturing(), cacheable = !recorded && !index.is_inference();
  const int64_t n = index.numel();
  if (cacheable) {
    std::lock_guard<std::mutex> lock(g_csr_mutex);
    for (auto it = g_csr.begin(); it != g_csr.end(); ++it) {
      if (it->nrows == nrows && it->version == index._version() && it->index.data_ptr() == index.data_ptr() && it->index.numel() == n &&
          it->index.scalar_type() == index.scalar_type() && it->index.device() == index.device()) {
        g_csr.splice(g_csr.begin(), g_csr, it);
        return {it->offsets, it->perm};
      }
    }
  }
  const c10::DeviceGuard guard(index.device());
  at::Tensor offsets = new_tensor({nrows + 1}, at::kLong, index.device()), perm = new_tensor({std::max<int64_t>(n, 1)}, at::kLong, index.device());
  const int64_t bytes = lib().cueq_segment_csr_workspace(n, nrows);
  at::Tensor ws = new_tensor({bytes}, at::kByte, index.device());
  std::optional<pybind11::gil_scoped_release> release;  // (the build waits for two flags)
  if (PyGILState_Check()) release.emplace();
  const auto build = recorded ? lib().cueq_segment_csr_build_async : lib().cueq_segment_csr_build;
  check(build(index.data_ptr(), index.scalar_type() == at::kLong ? 1 : 0, n, nrows, offsets.data_ptr<int64_t>(), perm.data_ptr<int64_t>(), ws.data_ptr(), bytes,
              stream_of(index.device().index())),
        "cueq_segment_csr_build");
  release.reset();
  if (cacheable) {
    // (the index tensor is kept alive with the entry so that its address cannot be reused meanwhile)
    std::list<CsrEntry> old;
    std::lock_guard<std::mutex> lock(g_csr_mutex);
    g_csr.push_front({index, offsets, perm, index._version(), nrows});
    if (g_csr.size() > 32) old.splice(old.begin(), g_csr, std::prev(g_csr.end()));
  }
  return {offsets, perm};
}

}  // namespace cueq_host

PYBIND11_MODULE(_host, m) {
  namespace py = pybind11;
  using namespace cueq_host;
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const CueqError& e) {
      PyErr_SetString(g_error_class ? g_error_class : PyExc_RuntimeError, e.what());
    }
  });
  m.def("load", &load);
  m.def("segment_csr", &segment_csr);
  m.def("executor", &executor);
  bind_uniform_1d(m);
  bind_triangle(m);
  bind_linear(m);
  bind_fully_connected(m);
  bind_rows(m);
}
