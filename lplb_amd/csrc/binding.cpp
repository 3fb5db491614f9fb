// Python entry points of the calls a serving loop makes per batch: argument checks, output tensors and the library
// call of CompiledSolver's plan, solve, solve_batched, count_idx and map_idx (_native.py) in native code.
//
// A batch's plan is one kernel of 8 us.  Checking nine tensors, allocating and handing 21 arguments to ctypes took the
// interpreter 5 of the 8.5 us that the calling thread needed for it, which a short batch then waited for.  Time of
// the calling thread per call, before -> with this file (the launch itself is 2.6 us of it): Planner.run 8.5 -> 5.6 us,
// plan 8.9 -> 5.4, solve_batched 6.8 -> 3.8, count_workload + solve_probs + weighted_select_target 25.9 -> 16.1.
// The library is reached through dlopen, so that this file needs nothing of it at link time.
#include <dlfcn.h>

#define PY_SSIZE_T_CLEAN
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/select.h>
#include <c10/hip/HIPStream.h>
#include <torch/version.h>

#include "../../include/lplb_hip.h"

namespace {

decltype(&lplb_last_error) last_error;
decltype(&lplb_plan) do_plan;
decltype(&lplb_solve_batched) do_solve_batched;
decltype(&lplb_solve) do_solve;
decltype(&lplb_count_idx) do_count_idx;
decltype(&lplb_map_idx) do_map_idx;
decltype(&lplb_map_idx_prepared) do_map_idx_prepared;
decltype(&lplb_prepared_mapping_bytes) prepared_bytes;
PyObject *unsupported_shape;

struct PythonErrorIsSet {};

void require(bool cond, const char *what) {
  if (!cond) {
    PyErr_Format(PyExc_RuntimeError, "LPLB assertion failed: %s", what);
    throw PythonErrorIsSet{};
  }
}
template <typename F> void call_library(F &&f) {   // other Python threads may run meanwhile
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  if (rc != LPLB_OK) {
    PyErr_Format(rc == LPLB_EUNSUPPORTED ? unsupported_shape : PyExc_RuntimeError, "lplb_hip error %d: %s", rc, last_error());
    throw PythonErrorIsSet{};
  }
}
const at::Tensor &tensor(PyObject *o, const char *name) {
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "%s must be a tensor, got %s", name, Py_TYPE(o)->tp_name);
    throw PythonErrorIsSet{};
  }
  return THPVariable_Unpack(o);
}
const at::Tensor *tensor_or_none(PyObject *o, const char *name) { return o == nullptr || o == Py_None ? nullptr : &tensor(o, name); }
int64_t integer(PyObject *o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred())
    throw PythonErrorIsSet{};
  return v;
}
bool is(const at::Tensor &t, at::ScalarType type) { return t.scalar_type() == type && t.is_cuda() && t.is_contiguous(); }
bool is_1d(const at::Tensor &t, int64_t n) { return t.dim() == 1 && t.size(0) == n; }
bool is_2d(const at::Tensor &t, int64_t n, int64_t m) { return t.dim() == 2 && t.size(0) == n && t.size(1) == m; }
int32_t *ints(const at::Tensor &t) { return static_cast<int32_t *>(t.data_ptr()); }
float *floats(const at::Tensor &t) { return static_cast<float *>(t.data_ptr()); }
int64_t *longs(const at::Tensor &t) { return static_cast<int64_t *>(t.data_ptr()); }
at::Tensor make(at::IntArrayRef shape, at::ScalarType type, const at::Tensor &like) {
  return at::detail::empty_cuda(shape, type, like.device(), std::nullopt);
}
lplb_stream_t stream_of(const at::Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
// What fits a signed 32-bit argument of the library is handed on; the rest it would have to refuse anyway.
int as_int(int64_t v) {
  require(v >= INT32_MIN && v <= INT32_MAX, "a number that fits 32 bits");
  return (int)v;
}

// The first seven arguments of every function: n_group, group_size, dup_per_rank, n_combined_experts, n_local_experts,
// step_rule, n_steps.
struct Shape {
  int n_group, G, D, C, P, step_rule, n_steps;
  int64_t n_experts;
  explicit Shape(PyObject *const *args) {
    int v[7];
    for (int i = 0; i < 7; ++i)
      v[i] = as_int(integer(args[i]));
    n_group = v[0]; G = v[1]; D = v[2]; C = v[3]; P = v[4]; step_rule = v[5]; n_steps = v[6];
    n_experts = (int64_t)(P - D * C) * G * n_group;
  }
};
constexpr Py_ssize_t kShapeArgs = 7;

template <typename F> PyObject *guarded(Py_ssize_t n_args, Py_ssize_t wanted, F &&f) {
  if (n_args != kShapeArgs + wanted) {
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", kShapeArgs + wanted, n_args);
    return nullptr;
  }
  HANDLE_TH_ERRORS
  try {
    return f();
  } catch (const PythonErrorIsSet &) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}
void check_physical_counts(const at::Tensor *t, const Shape &s) {
  require(t == nullptr || (is(*t, at::kInt) && t->numel() == (int64_t)s.n_group * s.G * s.P),
          "physical_counts is a contiguous int32 [n_group * group_size * n_local_experts] GPU tensor");
}
PyObject *pack(std::initializer_list<PyObject *> items) {   // takes the references
  PyObject *t = PyTuple_New((Py_ssize_t)items.size());
  Py_ssize_t i = 0;
  for (PyObject *o : items)
    PyTuple_SET_ITEM(t, i++, o);
  return t;
}
PyObject *wrapped(const at::Tensor &t) { return THPVariable_Wrap(t); }

// plan(shape..., idx, r2o, o2r, phy2log, avail_num, n_sms, global_counts, workspace, physical_counts)
PyObject *plan(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  return guarded(n_args, 9, [&]() -> PyObject * {
    const Shape s(args);
    args += kShapeArgs;
    const at::Tensor &idx = tensor(args[0], "idx"), &r2o = tensor(args[1], "r2o"), &o2r = tensor(args[2], "o2r"),
                     &phy2log = tensor(args[3], "phy2log"), &avail = tensor(args[4], "avail_num");
    const int n_sms = as_int(integer(args[5]));
    const at::Tensor *counts = tensor_or_none(args[6], "global_counts"), *physical = tensor_or_none(args[8], "physical_counts");
    require(is(idx, at::kLong), "idx is a contiguous int64 GPU tensor");
    require(is(r2o, at::kInt) && is_2d(r2o, s.G, s.D), "r2o is a contiguous int32 [group_size, dup_per_rank] GPU tensor");
    require(is(o2r, at::kInt) && is_2d(o2r, s.G, s.D), "o2r is a contiguous int32 [group_size, dup_per_rank] GPU tensor");
    require(is(phy2log, at::kInt) && is_1d(phy2log, (int64_t)s.G * s.n_group * s.P),
            "phy2log is a contiguous int32 [n_group * group_size * n_local_experts] GPU tensor");
    require(avail.numel() == 1 && avail.scalar_type() == at::kInt && avail.is_cuda(), "avail_num is one int32 on the GPU");
    require(!counts || (is(*counts, at::kInt) && counts->numel() == s.n_experts),
            "global_counts is a contiguous int32 [n_experts] GPU tensor");
    check_physical_counts(physical, s);
    // what the caller's dictionary, or any object with its `get` and `update`, keeps from batch to batch (never `out`,
    // unless the caller has put one there: that is the result)
    PyObject *ws = args[7] == Py_None ? nullptr : args[7];
    const bool is_dict = ws && PyDict_CheckExact(ws);
    THPObjectPtr got[4];
    int n_got = 0;
    auto kept = [&](const char *key) -> const at::Tensor * {
      if (!ws)
        return nullptr;
      if (is_dict)
        return tensor_or_none(PyDict_GetItemString(ws, key), key);
      THPObjectPtr &o = got[n_got++] = PyObject_CallMethod(ws, "get", "s", key);
      if (!o)
        throw PythonErrorIsSet{};
      return tensor_or_none(o.get(), key);
    };
    auto keep = [&](const char *key, PyObject *value) {
      if (!ws)
        return;
      if (is_dict) {
        if (PyDict_SetItemString(ws, key, value) < 0)
          throw PythonErrorIsSet{};
        return;
      }
      THPObjectPtr update(PyObject_GetAttrString(ws, "update")), none(PyTuple_New(0)), one(Py_BuildValue("{sO}", key, value));
      if (!update || !none || !one || !THPObjectPtr(PyObject_Call(update.get(), none.get(), one.get())))
        throw PythonErrorIsSet{};
    };
    const at::Tensor *k_out = kept("out"), *k_by_sm = kept("by_sm"), *k_weight = kept("o_weight"), *k_workload = kept("global_workload");
    // (kept for another shape or device: a new one takes its place)
    auto fits = [&](const at::Tensor *t, at::ScalarType type, int64_t numel) {
      return t && is(*t, type) && t->numel() == numel && t->device() == idx.device();
    };
    const int64_t n_shares = (int64_t)s.n_group * s.G * s.D;
    const bool new_table = !(fits(k_by_sm, at::kInt, n_sms * s.n_experts) && is_2d(*k_by_sm, n_sms, s.n_experts));
    const bool new_weight = !fits(k_weight, at::kFloat, n_shares), new_workload = !fits(k_workload, at::kFloat, s.n_experts);
    const at::Tensor out = fits(k_out, at::kLong, idx.numel()) && k_out->sizes() == idx.sizes() ? *k_out : make(idx.sizes(), at::kLong, idx);
    const at::Tensor by_sm = new_table ? make({n_sms, s.n_experts}, at::kInt, idx) : *k_by_sm;
    const at::Tensor weight = new_weight ? make({s.n_group, s.G, s.D}, at::kFloat, idx) : *k_weight;
    const at::Tensor workload = new_workload ? make({s.n_experts}, at::kFloat, idx) : *k_workload;
    THPObjectPtr py_by_sm(wrapped(by_sm)), py_weight(wrapped(weight));
    if (new_table)
      keep("by_sm", py_by_sm.get());
    if (new_weight)
      keep("o_weight", py_weight.get());
    if (new_workload)
      keep("global_workload", THPObjectPtr(wrapped(workload)).get());
    call_library([&] {
      return do_plan(longs(idx), idx.numel(), counts ? ints(*counts) : nullptr, ints(r2o), ints(o2r), ints(phy2log), s.n_group, s.G,
                     s.D, s.C, s.P, n_sms, ints(by_sm), floats(workload), floats(weight), ints(avail), longs(out),
                     physical ? ints(*physical) : nullptr, s.step_rule, s.n_steps, stream_of(idx));
    });
    return pack({wrapped(out), py_weight.release(), py_by_sm.release()});
  });
}

// solve(shape..., local_workload, r2o, phy2log, avail_num)
PyObject *solve(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  return guarded(n_args, 4, [&]() -> PyObject * {
    const Shape s(args);
    args += kShapeArgs;
    const at::Tensor &workload = tensor(args[0], "local_workload"), &avail = tensor(args[3], "avail_num");
    require(workload.is_cuda(), "local_workload on a GPU");
    require(workload.dim() == 3, "local_workload.dim() == 3");
    const int64_t n_group = workload.size(0), L = workload.size(2), n_pes = n_group * s.G;
    require(workload.size(1) == s.G, "group_size == local_workload.size(1)");
    require(workload.scalar_type() == at::kInt, "local_workload.dtype == int32");
    require(workload.is_contiguous(), "local_workload.is_contiguous()");
    const at::Tensor &r2o = tensor(args[1], "r2o"), &phy2log = tensor(args[2], "phy2log");
    require(is_2d(r2o, s.G, s.D), "r2o is [group_size, dup_per_rank]");
    require(r2o.scalar_type() == at::kInt, "r2o.dtype == int32");
    require(phy2log.dim() == 1 && n_pes > 0 && phy2log.size(0) % n_pes == 0, "phy2log is 1-D, a multiple of the EP size");
    require(phy2log.scalar_type() == at::kInt, "phy2log.dtype == int32");
    const int64_t replicas = phy2log.size(0) / n_pes - L;
    require(s.D > 0 && replicas % s.D == 0, "replicas per rank divisible by dup_per_rank");
    require(avail.numel() == 1, "avail_num.numel() == 1");
    require(avail.scalar_type() == at::kInt, "avail_num.dtype == int32");
    require(r2o.is_cuda() && phy2log.is_cuda() && avail.is_cuda(), "all tensors on the GPU");
    const at::Tensor r2o_c = r2o.contiguous(), phy2log_c = phy2log.contiguous();
    const at::Tensor global = make(workload.sizes(), at::kFloat, workload), result = make({n_group, s.G, s.D}, at::kFloat, workload);
    const int64_t per_var = replicas / s.D;
    call_library([&] {
      return do_solve(ints(workload), floats(global), ints(r2o_c), ints(phy2log_c), (int)n_group, s.G, s.D, (int)per_var,
                      (int)(L - s.D * per_var), ints(avail), floats(result), s.step_rule, s.n_steps, stream_of(workload));
    });
    return pack({wrapped(result), wrapped(global)});
  });
}

// solve_batched(shape..., workloads, r2o, phy2log, avail_num, want_global)
PyObject *solve_batched(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  return guarded(n_args, 5, [&]() -> PyObject * {
    const Shape s(args);
    args += kShapeArgs;
    const at::Tensor &workloads = tensor(args[0], "workloads"), &r2o = tensor(args[1], "r2o"), &phy2log = tensor(args[2], "phy2log"),
                     &avail = tensor(args[3], "avail_num");
    const bool want_global = PyObject_IsTrue(args[4]) == 1;
    require(is(workloads, at::kInt) && workloads.dim() == 4, "workloads is a contiguous int32 [N, n_group, G, L] GPU tensor");
    const int64_t n_inst = workloads.size(0), n_group = workloads.size(1), L = workloads.size(3), n_pes = n_group * s.G;
    require(workloads.size(2) == s.G, "group_size == workloads.size(2)");
    require(phy2log.scalar_type() == at::kInt && phy2log.dim() == 1 && n_pes > 0 && phy2log.size(0) % n_pes == 0,
            "phy2log is int32, 1-D, a multiple of the EP size");
    require(r2o.scalar_type() == at::kInt && is_2d(r2o, s.G, s.D), "r2o is int32 [G, D]");
    require(avail.numel() == 1 && avail.scalar_type() == at::kInt, "avail_num is one int32");
    require(r2o.is_cuda() && phy2log.is_cuda() && avail.is_cuda(), "all tensors on the GPU");
    require(s.D > 0, "dup_per_rank is positive");
    const int n_inst32 = as_int(n_inst);
    const int64_t per_var = (phy2log.size(0) / n_pes - L) / s.D;
    const at::Tensor r2o_c = r2o.contiguous(), phy2log_c = phy2log.contiguous();
    const at::Tensor result = make({n_inst, n_group, s.G, s.D}, at::kFloat, workloads);
    const at::Tensor global = want_global ? make(workloads.sizes(), at::kFloat, workloads) : at::Tensor();
    call_library([&] {
      return do_solve_batched(ints(workloads), want_global ? floats(global) : nullptr, ints(r2o_c), ints(phy2log_c), n_inst32,
                              (int)n_group, s.G, s.D, (int)per_var, (int)(L - s.D * per_var), ints(avail), floats(result),
                              s.step_rule, s.n_steps, stream_of(workloads));
    });
    return want_global ? pack({wrapped(result), wrapped(global)}) : wrapped(result);
  });
}

// count_idx(shape..., idx, n_sms, out)
PyObject *count_idx(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  return guarded(n_args, 3, [&]() -> PyObject * {
    const Shape s(args);
    args += kShapeArgs;
    const at::Tensor &idx = tensor(args[0], "idx");
    const int n_sms = as_int(integer(args[1]));
    const at::Tensor *given = tensor_or_none(args[2], "out");
    require(idx.scalar_type() == at::kLong, "idx.dtype == int64");
    require(idx.is_cuda(), "idx.device().is_cuda()");
    require(idx.is_contiguous(), "idx.is_contiguous()");
    require(!given || (is(*given, at::kInt) && is_2d(*given, n_sms, s.n_experts)),
            "out: int32 [n_sms, n_experts], contiguous, on the GPU");
    const at::Tensor out = given ? *given : make({n_sms, s.n_experts}, at::kInt, idx);
    const int n_experts = as_int(s.n_experts);
    call_library([&] { return do_count_idx(longs(idx), idx.numel(), n_experts, n_sms, ints(out), stream_of(idx)); });
    return pack({wrapped(at::select(out, 0, -1)), wrapped(out)});
  });
}

// map_idx(shape..., mapping_idx, o_weight, local_workload_split_by_sm, o2r, phy2log, n_sms, physical_counts, prepared)
PyObject *map_idx(PyObject *, PyObject *const *args, Py_ssize_t n_args) {
  return guarded(n_args, 8, [&]() -> PyObject * {
    const Shape s(args);
    args += kShapeArgs;
    const at::Tensor &idx = tensor(args[0], "mapping_idx"), &weight = tensor(args[1], "o_weight"),
                     &by_sm = tensor(args[2], "local_workload_split_by_sm"), &o2r = tensor(args[3], "o2r"),
                     &phy2log = tensor(args[4], "phy2log");
    const int n_sms = as_int(integer(args[5]));
    const at::Tensor *physical = tensor_or_none(args[6], "physical_counts"), *prepared = tensor_or_none(args[7], "prepared");
    require(idx.scalar_type() == at::kLong, "mapping_idx.dtype == int64");
    require(idx.is_cuda(), "mapping_idx.device().is_cuda()");
    require(idx.is_contiguous(), "mapping_idx.is_contiguous()");
    require(weight.scalar_type() == at::kFloat, "o_weight.dtype == float32");
    require(weight.is_cuda() && weight.is_contiguous(), "o_weight is a contiguous GPU tensor");
    require(weight.dim() == 3 && weight.size(0) == s.n_group && weight.size(1) == s.G && weight.size(2) == s.D,
            "o_weight is [n_group, group_size, dup_per_rank]");
    require(is(o2r, at::kInt), "o2r is a contiguous int32 GPU tensor");
    require(is_2d(o2r, s.G, s.D), "o2r is [group_size, dup_per_rank]");
    require(is(phy2log, at::kInt), "phy2log is a contiguous int32 GPU tensor");
    require(is_1d(phy2log, (int64_t)s.G * s.n_group * s.P), "phy2log.size(0) == group_size * n_group * n_local_experts");
    require(is(by_sm, at::kInt) && is_2d(by_sm, n_sms, s.n_experts),
            "local_workload_split_by_sm is a contiguous int32 [n_sms, n_experts] GPU tensor");
    check_physical_counts(physical, s);
    require(!prepared || (is(*prepared, at::kInt) && prepared->numel() * 4 >= prepared_bytes(s.n_group, s.G, s.D, s.C, s.P)),
            "prepared is a table from prepare_mapping");
    const at::Tensor out = make(idx.sizes(), at::kLong, idx);
    int32_t *counts = physical ? ints(*physical) : nullptr;
    call_library([&] {
      return prepared ? do_map_idx_prepared(longs(idx), floats(weight), ints(by_sm), ints(*prepared), idx.numel(), s.n_group, s.G, s.D,
                                            s.C, s.P, n_sms, longs(out), counts, stream_of(idx))
                      : do_map_idx(longs(idx), floats(weight), ints(by_sm), ints(o2r), ints(phy2log), idx.numel(), s.n_group, s.G,
                                   s.D, s.C, s.P, n_sms, longs(out), counts, stream_of(idx));
    });
    return wrapped(out);
  });
}

// bind(path of the library, exception for LPLB_EUNSUPPORTED)
PyObject *bind(PyObject *, PyObject *args) {
  const char *path = nullptr;
  PyObject *exception = nullptr;
  if (!PyArg_ParseTuple(args, "sO", &path, &exception))
    return nullptr;
  void *lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!lib) {
    PyErr_SetString(PyExc_RuntimeError, dlerror());
    return nullptr;
  }
  auto find = [&](auto &f, const char *name) {
    f = reinterpret_cast<std::remove_reference_t<decltype(f)>>(dlsym(lib, name));
    if (!f)
      PyErr_Format(PyExc_RuntimeError, "%s has no %s", path, name);
    return f != nullptr;
  };
  if (!(find(last_error, "lplb_last_error") && find(do_plan, "lplb_plan") && find(do_solve, "lplb_solve") &&
        find(do_solve_batched, "lplb_solve_batched") && find(do_count_idx, "lplb_count_idx") && find(do_map_idx, "lplb_map_idx") &&
        find(do_map_idx_prepared, "lplb_map_idx_prepared") && find(prepared_bytes, "lplb_prepared_mapping_bytes")))
    return nullptr;
  Py_INCREF(exception);
  Py_XDECREF(unsupported_shape);
  unsupported_shape = exception;
  Py_RETURN_NONE;
}

#define LPLB_FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, nullptr},
                         LPLB_FAST(plan), LPLB_FAST(solve), LPLB_FAST(solve_batched), LPLB_FAST(count_idx), LPLB_FAST(map_idx),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods};

} // namespace

PyMODINIT_FUNC PyInit__binding() {
  PyObject *m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
