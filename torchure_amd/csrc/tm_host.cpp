// tm_host.cpp -- host-side list primitives of the optimizer step (CPU only, no GPU work).
//
// The per-step host path walks every parameter: it gathers each grad, checks that the
// pointers cached in the tensor table are still the tensors' storage, compares autograd
// versions and bumps them after the raw-pointer writes. In Python each of those accesses
// costs 0.1-0.2 us per tensor, which for a list of 10,000 tensors adds up to tens of
// milliseconds per step. These functions do the same walks over Python lists in C++
// (about 15-20 ns per element), so the steady-state step stays far below the kernel time.
// They read tensor metadata only; nothing here allocates or touches device memory.

#include <torch/extension.h>
#include <pybind11/numpy.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/variable.h>

#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

namespace py = pybind11;

namespace {

// The attribute `name` of o, or nullptr when it has none or it is None (new reference otherwise).
// A missing attribute is looked up without raising: on a list of params without working copies
// the AttributeErrors took most of the walk (150 ns each).
PyObject* attr_or_null(PyObject* o, PyObject* name) {
  PyObject* a = nullptr;
  if (_PyObject_LookupAttr(o, name, &a) < 0) throw py::error_already_set();
  if (a == Py_None) Py_CLEAR(a);
  return a;
}

// nullptr for None; throws for anything that is not a tensor.
inline const at::Tensor* tensor_or_null(PyObject* o) {
  if (o == Py_None) return nullptr;
  if (!THPVariable_Check(o)) throw py::type_error("torchure_amd._tm_host: expected a tensor or None");
  return &THPVariable_Unpack(o);
}

inline PyObject* list_item(const py::list& l, Py_ssize_t i) { return PyList_GET_ITEM(l.ptr(), i); }

// Effective grad of each master: p.grad if set, else works[i].grad (works[i] may be None).
// Returns (list of grad tensors or None, bytes of sources: 0 none, 1 p.grad, 2 works[i].grad).
py::tuple grads(const py::list& params, const py::list& works) {
  const Py_ssize_t n = PyList_GET_SIZE(params.ptr());
  if (PyList_GET_SIZE(works.ptr()) != n) throw py::value_error("params and works differ in length");
  py::list out(n);
  std::string src(static_cast<size_t>(n), '\0');
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor* p = tensor_or_null(list_item(params, i));
    PyObject* g = nullptr;
    if (p && p->grad().defined()) {
      g = THPVariable_Wrap(p->grad());
      src[i] = 1;
    } else if (const at::Tensor* w = tensor_or_null(list_item(works, i)); w && w->grad().defined()) {
      g = THPVariable_Wrap(w->grad());
      src[i] = 2;
    }
    if (!g) {
      Py_INCREF(Py_None);
      g = Py_None;
    }
    PyList_SET_ITEM(out.ptr(), i, g);  // steals the reference
  }
  return py::make_tuple(out, py::bytes(src));
}

// data_ptr of each tensor (0 for None).
py::array_t<uint64_t> ptrs(const py::list& ts) {
  const Py_ssize_t n = PyList_GET_SIZE(ts.ptr());
  py::array_t<uint64_t> out(n);
  uint64_t* o = out.mutable_data();
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor* t = tensor_or_null(list_item(ts, i));
    o[i] = (t && t->defined()) ? reinterpret_cast<uint64_t>(t->data_ptr()) : 0u;
  }
  return out;
}

// Autograd version counter of each tensor (-1 for None).
py::array_t<int64_t> versions(const py::list& ts) {
  const Py_ssize_t n = PyList_GET_SIZE(ts.ptr());
  py::array_t<int64_t> out(n);
  int64_t* o = out.mutable_data();
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor* t = tensor_or_null(list_item(ts, i));
    o[i] = t ? static_cast<int64_t>(t->_version()) : -1;
  }
  return out;
}

// Sum of the version counters (versions only grow, so an in-place change raises it).
int64_t version_sum(const py::list& ts) {
  const Py_ssize_t n = PyList_GET_SIZE(ts.ptr());
  int64_t s = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor* t = tensor_or_null(list_item(ts, i));
    if (t) s += static_cast<int64_t>(t->_version());
  }
  return s;
}

// True if every entry is a dense (strided), contiguous tensor.
bool dense_contiguous(const py::list& ts) {
  const Py_ssize_t n = PyList_GET_SIZE(ts.ptr());
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor* t = tensor_or_null(list_item(ts, i));
    if (!t || !t->defined() || t->layout() != at::kStrided || !t->is_contiguous()) return false;
  }
  return true;
}

// True if both lists hold the same Python objects in the same order.
bool same(const py::list& a, const py::list& b) {
  const Py_ssize_t n = PyList_GET_SIZE(a.ptr());
  if (PyList_GET_SIZE(b.ptr()) != n) return false;
  for (Py_ssize_t i = 0; i < n; ++i)
    if (list_item(a, i) != list_item(b, i)) return false;
  return true;
}

// Grad-table fields of each tensor: (data_ptr uint64, numel int64, code uint8) with code 0
// for a dense contiguous bfloat16 tensor on a GPU, 1 for float32 likewise, 255 otherwise
// (the caller then reports the exact reason from Python).
py::tuple grad_fields(const py::list& ts) {
  const Py_ssize_t n = PyList_GET_SIZE(ts.ptr());
  py::array_t<uint64_t> ptr(n);
  py::array_t<int64_t> numel(n);
  py::array_t<uint8_t> code(n);
  uint64_t* pp = ptr.mutable_data();
  int64_t* pn = numel.mutable_data();
  uint8_t* pc = code.mutable_data();
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor* t = tensor_or_null(list_item(ts, i));
    const bool strided = t && t->defined() && t->layout() == at::kStrided;  // sparse ones have no data_ptr
    uint8_t c = 255;
    if (strided && t->is_cuda() && t->is_contiguous()) {
      const auto st = t->scalar_type();
      c = st == at::kBFloat16 ? 0 : (st == at::kFloat ? 1 : 255);
    }
    pc[i] = c;
    pp[i] = strided ? reinterpret_cast<uint64_t>(t->data_ptr()) : 0u;
    pn[i] = strided ? t->numel() : 0;
  }
  return py::make_tuple(ptr, numel, code);
}

// Lookup that does not run a defaultdict's factory: a missing entry is a mismatch below.
PyObject* dict_item(PyObject* d, PyObject* k) {  // borrowed, or nullptr if absent
  PyObject* r = PyDict_GetItemWithError(d, k);
  if (!r && PyErr_Occurred()) throw py::error_already_set();
  return r;
}

// True if every states[i] is a dict whose "exp_avg", "exp_avg_sq" and "step" entries are ms[i],
// vs[i] and ss[i] (object identity).
bool entries_same(const py::list& states, const py::list& ms, const py::list& vs, const py::list& ss) {
  const Py_ssize_t n = PyList_GET_SIZE(states.ptr());
  for (const py::list* l : {&ms, &vs, &ss})
    if (PyList_GET_SIZE(l->ptr()) != n) return false;
  static PyObject* k_m = PyUnicode_InternFromString("exp_avg");
  static PyObject* k_v = PyUnicode_InternFromString("exp_avg_sq");
  static PyObject* k_s = PyUnicode_InternFromString("step");
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* st = list_item(states, i);
    if (!PyDict_Check(st) || dict_item(st, k_m) != list_item(ms, i) || dict_item(st, k_v) != list_item(vs, i) ||
        dict_item(st, k_s) != list_item(ss, i))
      return false;
  }
  return true;
}

// The same, and state_map[params[i]] is states[i] for every i.
bool states_same(const py::dict& state_map, const py::list& params, const py::list& states,
                 const py::list& ms, const py::list& vs, const py::list& ss) {
  const Py_ssize_t n = PyList_GET_SIZE(params.ptr());
  if (PyList_GET_SIZE(states.ptr()) != n) return false;
  for (Py_ssize_t i = 0; i < n; ++i)
    if (dict_item(state_map.ptr(), list_item(params, i)) != list_item(states, i)) return false;
  return entries_same(states, ms, vs, ss);
}

// True if d holds exactly these key and value objects in this order. Compared in the dict's own
// order, so no key is hashed (a tensor's hash is a Python call, 0.2 us).
bool items_same(const py::dict& d, const py::list& keys, const py::list& values) {
  const Py_ssize_t n = PyList_GET_SIZE(keys.ptr());
  if (PyDict_Size(d.ptr()) != n || PyList_GET_SIZE(values.ptr()) != n) return false;
  PyObject *k, *v;
  Py_ssize_t pos = 0, i = 0;
  while (PyDict_Next(d.ptr(), &pos, &k, &v)) {
    if (i >= n || k != list_item(keys, i) || v != list_item(values, i)) return false;
    ++i;
  }
  return i == n;
}

// True if getattr(objs[i], name, None) is expected[i] for every i.
bool attrs_same(const py::list& objs, const py::str& name, const py::list& expected) {
  const Py_ssize_t n = PyList_GET_SIZE(objs.ptr());
  if (PyList_GET_SIZE(expected.ptr()) != n) return false;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* a = attr_or_null(list_item(objs, i), name.ptr());
    const bool same_obj = (a ? a : Py_None) == list_item(expected, i);
    Py_XDECREF(a);
    if (!same_obj) return false;
  }
  return true;
}

// Bumps the autograd version counter of every tensor, as an in-place op would.
void bump(const py::list& ts) {
  const Py_ssize_t n = PyList_GET_SIZE(ts.ptr());
  for (Py_ssize_t i = 0; i < n; ++i)
    if (const at::Tensor* t = tensor_or_null(list_item(ts, i))) torch::autograd::impl::bump_version(*t);
}

// Working-copy bookkeeping: works[i]._tm_master_version = params[i]._version and
// works[i]._tm_copy_version = works[i]._version, the versions read now. Views of one buffer
// share one counter, so a step that bumps several such masters raises each one's version by
// more than one: the versions are read back after the bumps rather than counted.
void stamp(const py::list& params, const py::list& works) {
  const Py_ssize_t n = PyList_GET_SIZE(params.ptr());
  if (PyList_GET_SIZE(works.ptr()) != n) throw py::value_error("params and works differ in length");
  static PyObject* k_master = PyUnicode_InternFromString("_tm_master_version");
  static PyObject* k_copy = PyUnicode_InternFromString("_tm_copy_version");
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor* p = tensor_or_null(list_item(params, i));
    const at::Tensor* w = tensor_or_null(list_item(works, i));
    if (!p || !w) throw py::value_error("torchure_amd._tm_host.stamp: None in a pair");
    for (auto [key, t] : {std::pair{k_master, p}, std::pair{k_copy, w}}) {
      PyObject* v = PyLong_FromLongLong(static_cast<long long>(t->_version()));
      if (!v) throw py::error_already_set();
      const int rc = PyObject_SetAttr(list_item(works, i), key, v);
      Py_DECREF(v);
      if (rc != 0) throw py::error_already_set();
    }
  }
}

// True if works[i]._tm_master_version equals params[i]._version for every i (the master has
// not been modified in place since its working copy was last written).
bool stamped(const py::list& params, const py::list& works) {
  const Py_ssize_t n = PyList_GET_SIZE(params.ptr());
  if (PyList_GET_SIZE(works.ptr()) != n) return false;
  static PyObject* k_master = PyUnicode_InternFromString("_tm_master_version");
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor* p = tensor_or_null(list_item(params, i));
    if (!p) return false;
    PyObject* a = PyObject_GetAttr(list_item(works, i), k_master);  // new reference
    if (!a) {
      if (!PyErr_ExceptionMatches(PyExc_AttributeError)) throw py::error_already_set();
      PyErr_Clear();
      return false;
    }
    const long long v = PyLong_Check(a) ? PyLong_AsLongLong(a) : -1;
    Py_DECREF(a);
    if (v == -1 && PyErr_Occurred()) PyErr_Clear();
    if (v != static_cast<long long>(p->_version())) return false;
  }
  return true;
}

PyObject* working_name() {
  static PyObject* name = PyUnicode_InternFromString("_tm_working");
  return name;
}

// For a clip over params: (grads, the params that carry them, their distinct `_tm_owner` marks).
// A master without a grad of its own contributes the grad of its working copy, if any.
py::tuple collect(const py::list& params) {
  static PyObject* k_owner = PyUnicode_InternFromString("_tm_owner");
  const Py_ssize_t n = PyList_GET_SIZE(params.ptr());
  py::list grads, holders, owners;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* po = list_item(params, i);
    const at::Tensor* p = tensor_or_null(po);
    if (!p) continue;
    py::object g;
    if (p->grad().defined()) {
      g = py::reinterpret_steal<py::object>(THPVariable_Wrap(p->grad()));
    } else {
      py::object wo = py::reinterpret_steal<py::object>(attr_or_null(po, working_name()));
      const at::Tensor* w = wo.ptr() ? tensor_or_null(wo.ptr()) : nullptr;
      if (!w || !w->grad().defined()) continue;
      g = py::reinterpret_steal<py::object>(THPVariable_Wrap(w->grad()));
    }
    grads.append(g);
    holders.append(py::reinterpret_borrow<py::object>(po));
    py::object own = py::reinterpret_steal<py::object>(attr_or_null(po, k_owner));
    if (!own.ptr()) own = py::none();
    bool known = false;
    for (const auto& o : owners) known = known || o.ptr() == own.ptr();
    if (!known) owners.append(own);
  }
  return py::make_tuple(grads, holders, owners);
}

// tm_tensor_t (include/torchure_amd.h) as the host writes it.
struct TensorRow {
  uint64_t master, exp_avg, exp_avg_sq, grad, param_bf16, step;
  int64_t numel;
  int32_t group;
  uint32_t flags;
};
static_assert(sizeof(TensorRow) == 64, "tm_tensor_t is 64 bytes");

// dtype code of a dense contiguous GPU grad (0 bfloat16, 1 float32), 255 for anything else.
inline uint8_t grad_code(const at::Tensor* t) {
  if (!t || !t->defined() || t->layout() != at::kStrided || !t->is_cuda() || !t->is_contiguous()) return 255;
  const auto st = t->scalar_type();
  return st == at::kBFloat16 ? 0 : (st == at::kFloat ? 1 : 255);
}

// The tensor table of a grad-only call: (bytes of n tm_tensor_t with grad, numel and flags set,
// numels, all usable, all on one device).
py::tuple grad_rows(const py::list& grads) {
  const Py_ssize_t n = PyList_GET_SIZE(grads.ptr());
  py::array_t<uint8_t> rows(static_cast<py::ssize_t>(n * sizeof(TensorRow)));
  py::array_t<int64_t> numels(n);
  TensorRow* r = reinterpret_cast<TensorRow*>(rows.mutable_data());
  int64_t* pn = numels.mutable_data();
  bool fine = true, one = true;
  c10::Device first(c10::kCPU);
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor* t = tensor_or_null(list_item(grads, i));
    const uint8_t code = grad_code(t);
    r[i] = TensorRow{};
    pn[i] = 0;
    if (!t || !t->defined()) {
      fine = false;
      continue;
    }
    if (i == 0) first = t->device();
    one = one && t->device() == first;
    fine = fine && code != 255;
    if (code == 255) continue;
    r[i].grad = reinterpret_cast<uint64_t>(t->data_ptr());
    r[i].numel = pn[i] = t->numel();
    r[i].flags = code;  // 0 = TM_GRAD_BF16, 1 = TM_GRAD_F32
  }
  return py::make_tuple(rows, numels, fine, one);
}

// The checks of the steady-state step in one walk: every param's working copy and grad source are
// the plan's, the grads dense and contiguous, the static tensors' pointers and the state dicts
// unchanged, and the working copies current. Returns (grads, their pointers), or None.
py::object plan_match(const py::list& all_params, const py::list& all_works, const py::bytes& src,
                      const py::list& statics, const py::array_t<uint64_t>& static_ptrs, const py::dict& state_map,
                      const py::list& state_keys, const py::list& state_values, const py::list& states,
                      const py::list& ms, const py::list& vs, const py::list& ss, const py::list& wparams,
                      const py::list& wworks) {
  const Py_ssize_t n = PyList_GET_SIZE(all_params.ptr());
  const char* want = PyBytes_AS_STRING(src.ptr());
  if (PyBytes_GET_SIZE(src.ptr()) != n ||
      !attrs_same(all_params, py::reinterpret_borrow<py::str>(working_name()), all_works))
    return py::none();
  py::list out;
  std::vector<uint64_t> at_ptr;
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor* p = tensor_or_null(list_item(all_params, i));
    const at::Tensor* w = tensor_or_null(list_item(all_works, i));
    const at::Tensor* g = nullptr;
    char from = 0;
    if (p && p->grad().defined()) {
      g = &p->grad();
      from = 1;
    } else if (w && w->grad().defined()) {
      g = &w->grad();
      from = 2;
    }
    if (from != want[i]) return py::none();
    if (!g) continue;
    if (g->layout() != at::kStrided || !g->is_contiguous()) return py::none();
    at_ptr.push_back(reinterpret_cast<uint64_t>(g->data_ptr()));
    out.append(py::reinterpret_steal<py::object>(THPVariable_Wrap(*g)));
  }
  const Py_ssize_t k = PyList_GET_SIZE(statics.ptr());
  if (static_ptrs.size() != k) return py::none();
  const uint64_t* sp = static_ptrs.data();
  for (Py_ssize_t i = 0; i < k; ++i) {
    const at::Tensor* t = tensor_or_null(list_item(statics, i));
    if (((t && t->defined()) ? reinterpret_cast<uint64_t>(t->data_ptr()) : 0u) != sp[i]) return py::none();
  }
  if (!items_same(state_map, state_keys, state_values) || !entries_same(states, ms, vs, ss)) return py::none();
  if (PyList_GET_SIZE(wparams.ptr()) && !stamped(wparams, wworks)) return py::none();
  py::array_t<uint64_t> ptrs_out(static_cast<py::ssize_t>(at_ptr.size()));
  std::copy(at_ptr.begin(), at_ptr.end(), ptrs_out.mutable_data());
  return py::make_tuple(out, ptrs_out);
}

// The params a clip measured and their grads against the plan's: every grad of the record, taken
// in the plan's order (perm), is the grad at hand, and none changed in place since.
// 0: other grads, 1: the same, 2: the same but modified.
int clip_match(const py::list& rec_grads, const std::vector<int64_t>& perm, const py::list& grads, int64_t total) {
  const Py_ssize_t n = PyList_GET_SIZE(grads.ptr());
  if (static_cast<Py_ssize_t>(perm.size()) != n) return 0;
  int64_t sum = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (perm[i] < 0 || perm[i] >= PyList_GET_SIZE(rec_grads.ptr())) return 0;
    if (list_item(rec_grads, perm[i]) != list_item(grads, i)) return 0;
    sum += static_cast<int64_t>(tensor_or_null(list_item(grads, i))->_version());
  }
  return sum == total ? 1 : 2;
}

// tm_accum_t (include/torchure_amd.h) as the host writes it.
struct AccumRow {
  uint64_t acc, micro;
  int64_t numel, flags;
};
static_assert(sizeof(AccumRow) == 32, "tm_accum_t is 32 bytes");

// One micro-step of accumulation over params: checks every param, its accumulator (p.grad) and
// its working copy's grad, then, only if all are usable, gives first micro-steps their
// accumulator (unfilled: the kernel assigns it). Returns (accumulators, those with a micro grad,
// rows, numels, the working copies' grads, device index), or None when the caller's checks should
// report why not (or there is nothing to do). None too where a param with a micro grad stands in
// the list more than once: its rows would write one accumulator from several workgroups of a launch.
py::object accumulate_scan(const py::list& params, bool last, int64_t assign_flag) {
  const Py_ssize_t n = PyList_GET_SIZE(params.ptr());
  struct Item {
    const at::Tensor *p, *w;
  };
  std::vector<Item> todo;
  std::vector<py::object> keep;  // the working copies, alive while their pointers are used
  std::vector<const void*> written;  // the params whose accumulator the launch writes
  c10::Device first(c10::kCPU);
  auto dense = [](const at::Tensor& t) { return t.layout() == at::kStrided && t.is_cuda() && t.is_contiguous(); };
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* po = list_item(params, i);
    const at::Tensor* p = tensor_or_null(po);
    if (!p) return py::none();
    py::object wo = py::reinterpret_steal<py::object>(attr_or_null(po, working_name()));
    const at::Tensor* w = wo.ptr() ? tensor_or_null(wo.ptr()) : nullptr;
    if (w && !w->grad().defined()) w = nullptr;
    const at::Tensor& g = p->grad();
    if (!w && (!last || !g.defined())) continue;
    if (!dense(*p) || (g.defined() ? g : *p).scalar_type() != at::kFloat || (g.defined() && !dense(g)))
      return py::none();
    if (w) {
      const at::Tensor& m = w->grad();
      if (!dense(m) || m.scalar_type() != at::kBFloat16 || m.numel() != p->numel() || m.device() != p->device())
        return py::none();
    }
    if (todo.empty()) first = p->device();
    if (p->device() != first) return py::none();
    todo.push_back({p, w});
    keep.push_back(wo);
    if (w) written.push_back(p->unsafeGetTensorImpl());
  }
  if (todo.empty()) return py::none();
  std::sort(written.begin(), written.end());
  if (std::adjacent_find(written.begin(), written.end()) != written.end()) return py::none();
  const py::ssize_t k = static_cast<py::ssize_t>(todo.size());
  py::array_t<uint8_t> rows(k * static_cast<py::ssize_t>(sizeof(AccumRow)));
  py::array_t<int64_t> numels(k);
  AccumRow* r = reinterpret_cast<AccumRow*>(rows.mutable_data());
  py::list accs(k), changed, micros;
  for (py::ssize_t i = 0; i < k; ++i) {
    const at::Tensor* p = todo[i].p;
    const at::Tensor* w = todo[i].w;
    const bool fresh = !p->grad().defined();
    if (fresh) {
      at::NoGradGuard no_grad;
      p->mutable_grad() = at::empty(p->sizes(), p->options().requires_grad(false));
    }
    const at::Tensor& g = p->grad();
    r[i] = AccumRow{reinterpret_cast<uint64_t>(g.data_ptr()), w ? reinterpret_cast<uint64_t>(w->grad().data_ptr()) : 0u,
                    g.numel(), fresh ? assign_flag : 0};
    numels.mutable_data()[i] = g.numel();
    PyObject* acc = THPVariable_Wrap(g);
    if (w) {
      changed.append(py::reinterpret_borrow<py::object>(acc));
      micros.append(py::reinterpret_steal<py::object>(THPVariable_Wrap(w->grad())));
    }
    PyList_SET_ITEM(accs.ptr(), i, acc);  // steals the reference
  }
  return py::make_tuple(accs, changed, rows, numels, micros, static_cast<int>(first.index()));
}

// Drops the grad of every param's working copy.
void clear_work_grads(const py::list& params) {
  const Py_ssize_t n = PyList_GET_SIZE(params.ptr());
  for (Py_ssize_t i = 0; i < n; ++i) {
    py::object wo = py::reinterpret_steal<py::object>(attr_or_null(list_item(params, i), working_name()));
    if (!wo.ptr()) continue;
    const at::Tensor* w = tensor_or_null(wo.ptr());
    if (w && w->grad().defined()) w->mutable_grad().reset();
  }
}

// Which tensors, at which versions: matches() tells whether a list holds exactly these tensors,
// unmodified since. Holds them weakly.
struct Stamp {
  std::vector<std::pair<c10::weak_intrusive_ptr<c10::TensorImpl>, int64_t>> seen;
  explicit Stamp(const py::list& ts) {
    const Py_ssize_t n = PyList_GET_SIZE(ts.ptr());
    seen.reserve(static_cast<size_t>(n));
    for (Py_ssize_t i = 0; i < n; ++i) {
      const at::Tensor* t = tensor_or_null(list_item(ts, i));
      if (!t) throw py::value_error("torchure_amd._tm_host.Stamp: expected tensors");
      seen.emplace_back(t->getIntrusivePtr(), static_cast<int64_t>(t->_version()));
    }
  }
  bool matches(const py::list& ts) const {
    const Py_ssize_t n = PyList_GET_SIZE(ts.ptr());
    if (static_cast<size_t>(n) != seen.size()) return false;
    for (Py_ssize_t i = 0; i < n; ++i) {
      const at::Tensor* t = tensor_or_null(list_item(ts, i));
      // a tensor that died and another at its address: the weak reference has expired
      if (!t || seen[i].first.expired() || seen[i].first._unsafe_get_target() != t->unsafeGetTensorImpl() ||
          static_cast<int64_t>(t->_version()) != seen[i].second)
        return false;
    }
    return true;
  }
};

}  // namespace

void tm_ce_host_bind(py::module_& m);  // tm_ce_host.cpp

PYBIND11_MODULE(_tm_host, m) {
  m.doc() = "torchure_amd host-side list primitives (CPU only)";
  tm_ce_host_bind(m);
  m.def("collect", &collect, "(grads, their params, distinct owner marks) of a list of params");
  m.def("grad_rows", &grad_rows, "tensor table of a grad-only call");
  m.def("plan_match", &plan_match, "the steady-state step's checks: (grads, pointers) or None");
  m.def("clip_match", &clip_match, "whether a clip's grads are the step's grads, unmodified");
  m.def("accumulate_scan", &accumulate_scan, "checks and table of one accumulation micro-step, or None");
  m.def("clear_work_grads", &clear_work_grads, "drop the grads of the params' working copies");
  py::class_<Stamp>(m, "Stamp", "tensors and their versions, held weakly")
      .def(py::init<const py::list&>())
      .def("matches", &Stamp::matches);
  m.def("grads", &grads, "effective grad per master (p.grad or its working copy's grad)");
  m.def("ptrs", &ptrs, "data_ptr of each tensor (0 for None)");
  m.def("versions", &versions, "autograd version of each tensor (-1 for None)");
  m.def("version_sum", &version_sum, "sum of autograd versions");
  m.def("dense_contiguous", &dense_contiguous, "all dense and contiguous");
  m.def("same", &same, "element-wise object identity of two lists");
  m.def("bump", &bump, "bump the autograd version of each tensor");
  m.def("stamp", &stamp, "record each master's and working copy's current version on the copy");
  m.def("stamped", &stamped, "every working copy's recorded master version is the master's current one");
  m.def("grad_fields", &grad_fields, "(data_ptr, numel, dtype code) of each grad");
  m.def("states_same", &states_same, "optimizer state dicts and their tensors are the given objects");
  m.def("attrs_same", &attrs_same, "getattr(obj, name, None) of each object is the given object");
}
