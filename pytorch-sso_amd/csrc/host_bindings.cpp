// Host side of the engine calls, without a Python loop over the tensors of a call: tables of
// device addresses, sizes and coefficients as the C ABI takes them (packed into bytes objects,
// which ctypes hands over as they are), the tensors of a factor product written into its job, and
// the order between two streams.
//
// A tensor is taken if it is a contiguous float32 tensor on a HIP device.  Where one is not, the
// functions return None (or False) and the caller finds out which and raises; nothing is launched here.
#include <hip/hip_runtime.h>
#include <torch/csrc/autograd/python_variable.h>

#include <map>
#include <mutex>

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
    {"order", KFAC_FAST(order), "order(device, waiting stream, stream waited for)"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
