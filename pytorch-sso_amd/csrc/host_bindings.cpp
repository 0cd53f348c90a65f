// Host side of the engine calls, without a Python loop over the tensors of a call: tables of
// device addresses, sizes and coefficients as the C ABI takes them (packed into bytes objects,
// which ctypes hands over as they are), the tensors of a factor product written into its job, and
// the order between two streams.
//
// A tensor is taken if it is a contiguous float32 tensor on a HIP device.  Where one is not, the
// functions return None (or False) and the caller finds out which and raises; nothing is launched here.
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>
#include <map>
#include <mutex>
#include <vector>

#include "../../include/kfac_hip.h"

namespace {

// address of a tensor the engine can take, or nullptr
void* address_of(PyObject* o) {
  if (!THPVariable_Check(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda() || t.scalar_type() != at::kFloat || t.layout() != at::kStrided || !t.is_contiguous())
    return nullptr;
  // (as Tensor.data_ptr(): a lazily copied tensor gets memory of its own before it is written to)
  return t.mutable_data_ptr();
}

// `fill(object, index, slot)` for every object of a list or tuple, into a bytes object of T; None where it
// returns false
template <class T, class FILL>
PyObject* packed(PyObject* list, FILL&& fill) {
  PyObject* const seq = PySequence_Fast(list, "expected a list or tuple");
  if (!seq) return nullptr;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
  PyObject* const bytes = PyBytes_FromStringAndSize(nullptr, n * (Py_ssize_t)sizeof(T));
  if (!bytes) {
    Py_DECREF(seq);
    return nullptr;
  }
  char* at = PyBytes_AS_STRING(bytes);
  bool ok = true;
  for (Py_ssize_t i = 0; ok && i < n; ++i, at += sizeof(T)) {
    T value{};
    ok = fill(PySequence_Fast_GET_ITEM(seq, i), value);
    memcpy(at, &value, sizeof(T));
  }
  Py_DECREF(seq);
  if (ok) return bytes;
  Py_DECREF(bytes);
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

// (exceptions of tensors without memory of their own, of sizes that are not known, ...: the caller's
// Python path raises them once more)
template <class F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (const std::exception&) {
    if (PyErr_Occurred()) PyErr_Clear();
    Py_RETURN_NONE;
  }
}

PyObject* pointer(PyObject*, PyObject* o) {
  return guarded([&]() -> PyObject* {
    void* const p = address_of(o);
    if (p == nullptr) Py_RETURN_NONE;
    return PyLong_FromVoidPtr(p);
  });
}

PyObject* pointers(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 2) {
    PyErr_SetString(PyExc_TypeError, "pointers(tensors, allow_none)");
    return nullptr;
  }
  const int allow_none = PyObject_IsTrue(args[1]);
  if (allow_none < 0) return nullptr;
  return guarded([&]() {
    return packed<void*>(args[0], [&](PyObject* o, void*& slot) {
      if (o == Py_None) return allow_none != 0;
      slot = address_of(o);
      return slot != nullptr;
    });
  });
}

PyObject* numels(PyObject*, PyObject* list) {
  return guarded([&]() {
    return packed<int64_t>(list, [](PyObject* o, int64_t& slot) {
      if (!THPVariable_Check(o)) return false;
      slot = THPVariable_Unpack(o).numel();
      return true;
    });
  });
}

template <class T>
PyObject* integers(PyObject*, PyObject* list) {
  return packed<T>(list, [](PyObject* o, T& slot) {
    const long long v = PyLong_AsLongLong(o);
    slot = (T)v;
    return !(v == -1 && PyErr_Occurred()) && (long long)slot == v;
  });
}

PyObject* floats(PyObject*, PyObject* list) {
  return packed<float>(list, [](PyObject* o, float& slot) {
    const double v = PyFloat_AsDouble(o);
    slot = (float)v;
    return !(v == -1. && PyErr_Occurred());
  });
}

// The elements of some lists of equal lengths, side by side
struct Columns {
  std::vector<PyObject*> lists;          // (as PySequence_Fast gives them)
  Py_ssize_t n = 0;
  bool ok = true;
  Columns(PyObject* const* args, int count) {
    for (int i = 0; i < count && ok; ++i) {
      PyObject* const seq = PySequence_Fast(args[i], "expected a list or tuple");
      if (!seq) {
        ok = false;
        return;
      }
      lists.push_back(seq);
      if (i == 0) n = PySequence_Fast_GET_SIZE(seq);
      else if (PySequence_Fast_GET_SIZE(seq) != n) ok = false;
    }
  }
  ~Columns() {
    for (PyObject* l : lists) Py_DECREF(l);
  }
  PyObject* at(int list, Py_ssize_t i) const { return PySequence_Fast_GET_ITEM(lists[list], i); }
};
const at::Tensor* tensor_of(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }
PyObject* int_list(const std::vector<int64_t>& v) {
  PyObject* const l = PyList_New((Py_ssize_t)v.size());
  if (!l) return nullptr;
  for (size_t i = 0; i < v.size(); ++i) {
    PyObject* const x = PyLong_FromLongLong(v[i]);
    if (!x) {
      Py_DECREF(l);
      return nullptr;
    }
    PyList_SET_ITEM(l, (Py_ssize_t)i, x);
  }
  return l;
}

// square_dims(tensors) -> their sizes, or None where one is no square matrix
PyObject* square_dims(PyObject*, PyObject* list) {
  return guarded([&]() -> PyObject* {
    const Columns c(&list, 1);
    if (!c.ok) return nullptr;
    std::vector<int64_t> dims;
    for (Py_ssize_t i = 0; i < c.n; ++i) {
      const at::Tensor* const t = tensor_of(c.at(0, i));
      if (!t || t->dim() != 2 || t->size(0) != t->size(1)) Py_RETURN_NONE;
      dims.push_back(t->size(0));
    }
    return int_list(dims);
  });
}

// outputs_fit(xs, firsts, seconds, exactly one) -> is there, for every x, a first output (with `exactly
// one`: either of the two and not both), and are the outputs of x's shape
PyObject* outputs_fit(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4) {
    PyErr_SetString(PyExc_TypeError, "outputs_fit(xs, firsts, seconds, exactly_one)");
    return nullptr;
  }
  const int exactly_one = PyObject_IsTrue(args[3]);
  if (exactly_one < 0) return nullptr;
  return guarded([&]() -> PyObject* {
    const Columns c(args, 3);
    if (PyErr_Occurred()) return nullptr;
    if (!c.ok) Py_RETURN_FALSE;
    for (Py_ssize_t i = 0; i < c.n; ++i) {
      const at::Tensor* const x = tensor_of(c.at(0, i));
      if (!x) Py_RETURN_FALSE;
      bool have[2];
      for (int k = 0; k < 2; ++k) {
        PyObject* const o = c.at(1 + k, i);
        have[k] = o != Py_None;
        const at::Tensor* const t = have[k] ? tensor_of(o) : nullptr;
        if (have[k] && (!t || t->sizes() != x->sizes())) Py_RETURN_FALSE;
      }
      if (exactly_one ? have[0] == have[1] : !have[0]) Py_RETURN_FALSE;
    }
    Py_RETURN_TRUE;
  });
}

// kron_dims(Ls, Rs, Ws, bs) -> (dG, dA) of layers whose weight- and bias-shaped tensors fit their factors, or None
PyObject* kron_dims(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4) {
    PyErr_SetString(PyExc_TypeError, "kron_dims(Ls, Rs, Ws, bs)");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    const Columns c(args, 4);
    if (PyErr_Occurred()) return nullptr;
    if (!c.ok) Py_RETURN_NONE;
    std::vector<int64_t> dG, dA;
    for (Py_ssize_t i = 0; i < c.n; ++i) {
      const at::Tensor *const L = tensor_of(c.at(0, i)), *const R = tensor_of(c.at(1, i)),
                       *const W = tensor_of(c.at(2, i));
      const bool bias = c.at(3, i) != Py_None;
      const at::Tensor* const b = bias ? tensor_of(c.at(3, i)) : nullptr;
      if (!L || !R || !W || (bias && !b) || L->dim() < 1 || R->dim() < 1 || W->dim() < 1) Py_RETURN_NONE;
      const int64_t g = L->size(0), a = R->size(0);
      if (W->numel() != g * (a - (bias ? 1 : 0)) || W->size(0) != g || (b && b->numel() != g)) Py_RETURN_NONE;
      dG.push_back(g);
      dA.push_back(a);
    }
    PyObject* const l = int_list(dG);
    PyObject* const r = l ? int_list(dA) : nullptr;
    PyObject* const both = r ? PyTuple_Pack(2, l, r) : nullptr;
    Py_XDECREF(l);
    Py_XDECREF(r);
    return both;
  });
}

// rowsq_sum(address of kfac_rowsq_sum, x, channels, scale or None, shift or None) -> the sums, or None
// where x is not what the engine takes as it is
PyObject* rowsq_sum(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 5) {
    PyErr_SetString(PyExc_TypeError, "rowsq_sum(function, x, channels, scale, shift)");
    return nullptr;
  }
  const auto run = (decltype(&kfac_rowsq_sum))PyLong_AsVoidPtr(args[0]);
  const long long channels = PyLong_AsLongLong(args[2]);
  if (PyErr_Occurred()) return nullptr;
  return guarded([&]() -> PyObject* {
    const float* const x = (const float*)address_of(args[1]);
    const float* const scale = args[3] == Py_None ? nullptr : (const float*)address_of(args[3]);
    const float* const shift = args[4] == Py_None ? nullptr : (const float*)address_of(args[4]);
    if (!run || !x || (args[3] != Py_None && !scale) || (args[4] != Py_None && !shift)) Py_RETURN_NONE;
    const at::Tensor& t = THPVariable_Unpack(args[1]);
    if (t.dim() < 2 || channels <= 0 || channels > INT_MAX || t.size(1) != channels || t.size(0) <= 0) Py_RETURN_NONE;
    const int64_t rows = t.size(0) * channels, len = t.numel() / rows;
    if (len <= 0 || len > INT_MAX) Py_RETURN_NONE;
    const at::Tensor out = at::empty({t.size(0), (int64_t)channels}, t.options().requires_grad(false));
    float* const sums = out.mutable_data_ptr<float>();
    const hipStream_t stream = c10::hip::getCurrentHIPStream(t.device().index()).stream();
    int status;
    // (a launch may wait for room in the stream's queue: other threads go on meanwhile)
    Py_BEGIN_ALLOW_THREADS
    status = run(x, rows, (int)channels, (int)len, scale, shift, sums, stream);
    Py_END_ALLOW_THREADS
    if (status != KFAC_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(out);
  });
}

// vectors(tensor, size, count) -> `count` new float32 vectors on the tensor's device
PyObject* vectors(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 3 || !THPVariable_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "vectors(tensor, size, count)");
    return nullptr;
  }
  const long long size = PyLong_AsLongLong(args[1]);
  const long count = PyLong_AsLong(args[2]);
  if (PyErr_Occurred()) return nullptr;
  return guarded([&]() -> PyObject* {
    const auto options = at::TensorOptions().dtype(at::kFloat).device(THPVariable_Unpack(args[0]).device());
    PyObject* const l = PyList_New(count);
    if (!l) return nullptr;
    for (long i = 0; i < count; ++i) {
      PyObject* const t = THPVariable_Wrap(at::empty({(int64_t)size}, options));
      if (!t) {
        Py_DECREF(l);
        return nullptr;
      }
      PyList_SET_ITEM(l, i, t);
    }
    return l;
  });
}

// update_job(address of a kfac_factor_job, x, out, prev or None, alpha, beta) -> done
PyObject* update_job(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 6) {
    PyErr_SetString(PyExc_TypeError, "update_job(job, x, out, prev, alpha, beta)");
    return nullptr;
  }
  kfac_factor_job* const job = (kfac_factor_job*)PyLong_AsVoidPtr(args[0]);
  const double alpha = PyFloat_AsDouble(args[4]), beta = PyFloat_AsDouble(args[5]);
  if (PyErr_Occurred()) return nullptr;
  bool ok = false;
  PyObject* const r = guarded([&]() -> PyObject* {
    void* const x = address_of(args[1]);
    void* const out = address_of(args[2]);
    void* const prev = args[3] == Py_None ? nullptr : address_of(args[3]);
    if (!job || !x || !out || (args[3] != Py_None && !prev)) Py_RETURN_NONE;
    job->x = (const float*)x;
    job->C = (float*)out;
    job->C_prev = (const float*)(prev ? prev : beta != 0. ? out : nullptr);
    job->alpha = (float)alpha;
    job->beta = (float)beta;
    ok = true;
    Py_RETURN_NONE;
  });
  Py_XDECREF(r);
  return PyBool_FromLong(ok);
}

// jobs(list of addresses) -> the jobs one behind the other
PyObject* jobs(PyObject*, PyObject* list) {
  return packed<kfac_factor_job>(list, [](PyObject* o, kfac_factor_job& slot) {
    const void* const p = PyLong_AsVoidPtr(o);
    if (!p) return false;
    slot = *(const kfac_factor_job*)p;
    return true;
  });
}

// order(device, waiting stream, stream waited for): what the first is given from now on runs behind what
// the second holds now.  One event per device serves all such orders: a wait refers to the record
// before it, whatever is recorded later.  (Never destroyed: no teardown order.)
std::mutex order_mutex;
std::map<int, hipEvent_t> order_events;

PyObject* order(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 3) {
    PyErr_SetString(PyExc_TypeError, "order(device, waiting, waited)");
    return nullptr;
  }
  const long device = PyLong_AsLong(args[0]);
  const hipStream_t waiting = (hipStream_t)PyLong_AsVoidPtr(args[1]);
  const hipStream_t waited = (hipStream_t)PyLong_AsVoidPtr(args[2]);
  if (PyErr_Occurred()) return nullptr;
  if (waiting == waited) Py_RETURN_NONE;
  hipError_t e = hipSuccess;
  {
    const std::lock_guard<std::mutex> lock(order_mutex);
    int current = -1;
    e = hipGetDevice(&current);
    if (e == hipSuccess && current != (int)device) e = hipSetDevice((int)device);
    hipEvent_t& event = order_events[(int)device];
    if (e == hipSuccess && event == nullptr) e = hipEventCreateWithFlags(&event, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventRecord(event, waited);
    if (e == hipSuccess) e = hipStreamWaitEvent(waiting, event, 0);
    if (current >= 0 && current != (int)device) (void)hipSetDevice(current);
  }
  if (e != hipSuccess) {
    PyErr_Format(PyExc_RuntimeError, "order of two streams: %s", hipGetErrorString(e));
    return nullptr;
  }
  Py_RETURN_NONE;
}

#define KFAC_FAST(f) (PyCFunction)(void (*)(void))(f), METH_FASTCALL
PyMethodDef methods[] = {
    {"pointer", pointer, METH_O, "device address of a tensor, or None"},
    {"pointers", KFAC_FAST(pointers), "pointers(tensors, allow_none): device addresses, or None"},
    {"numels", numels, METH_O, "number of elements of each tensor (int64)"},
    {"ints", integers<int>, METH_O, "int32 values"},
    {"int64s", integers<int64_t>, METH_O, "int64 values"},
    {"floats", floats, METH_O, "float32 values"},
    {"update_job", KFAC_FAST(update_job), "update_job(job, x, out, prev, alpha, beta)"},
    {"jobs", jobs, METH_O, "factor jobs by address, one behind the other"},
    {"square_dims", square_dims, METH_O, "sizes of square matrices, or None"},
    {"outputs_fit", KFAC_FAST(outputs_fit), "outputs_fit(xs, firsts, seconds, exactly_one)"},
    {"kron_dims", KFAC_FAST(kron_dims), "kron_dims(Ls, Rs, Ws, bs): (dG, dA), or None"},
    {"rowsq_sum", KFAC_FAST(rowsq_sum), "rowsq_sum(function, x, channels, scale, shift): the sums, or None"},
    {"vectors", KFAC_FAST(vectors), "vectors(tensor, size, count): new vectors on its device"},
    {"order", KFAC_FAST(order), "order(device, waiting stream, stream waited for)"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
