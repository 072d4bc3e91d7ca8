// Python extension module `akg_amd._launch`: the checks and the argument packing of a launch on device tensors, without
// the interpreter in between. A launch of a kernel of a few microseconds takes the time of its host call: written in Python
// (attribute reads per tensor, ctypes arrays, a torch.cuda.Stream object per call) 7.4 us, of which the launch itself 3.2.
//
// Both functions return None where anything is not as the fast path expects it (a wrong type, a check that fails, an
// exception): the caller then takes the Python path, which says what is wrong.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "../../include/akg_hip.h"

namespace {

PyObject *g_isCuda, *g_isContiguous, *g_nbytes, *g_dataPtr, *g_cudaStream;   // interned names

PyObject *notServed() {
  PyErr_Clear();
  Py_RETURN_NONE;
}

bool isTrue(PyObject *o) {   // takes the reference
  const bool r = o == Py_True;
  Py_XDECREF(o);
  return r;
}

// Address of a tensor that is a contiguous device tensor of `bytes` bytes; false otherwise.
bool tensorAddress(PyObject *t, PyObject *bytes, void **out) {
  if (!isTrue(PyObject_GetAttr(t, g_isCuda)) || !isTrue(PyObject_CallMethodNoArgs(t, g_isContiguous))) return false;
  PyObject *n = PyObject_GetAttr(t, g_nbytes);
  if (n == nullptr) return false;
  const int same = PyObject_RichCompareBool(n, bytes, Py_EQ);
  Py_DECREF(n);
  if (same != 1) return false;
  PyObject *p = PyObject_CallMethodNoArgs(t, g_dataPtr);
  if (p == nullptr) return false;
  *out = PyLong_AsVoidPtr(p);
  Py_DECREF(p);
  return !PyErr_Occurred();
}

bool pointerOf(PyObject *o, void **out) {
  if (!PyLong_CheckExact(o)) return false;
  *out = PyLong_AsVoidPtr(o);
  return !PyErr_Occurred();
}

// launch(handle, nbytes, tensors, stream, get_device, get_raw_stream) -> return code or None
PyObject *launch(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (nargs != 6 || !PyTuple_CheckExact(args[1]) || !(PyList_CheckExact(args[2]) || PyTuple_CheckExact(args[2]))) Py_RETURN_NONE;
  const Py_ssize_t n = PyTuple_GET_SIZE(args[1]);
  void *handle = nullptr, *stream = nullptr;
  void *ptrs[64];
  if (n > 64 || PySequence_Fast_GET_SIZE(args[2]) != n || !pointerOf(args[0], &handle)) return notServed();
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (PySequence_Fast_GET_SIZE(args[2]) != n) return notServed();   // (changed by what an attribute ran)
    PyObject *t = PySequence_Fast_GET_ITEM(args[2], i);
    Py_INCREF(t);
    const bool ok = tensorAddress(t, PyTuple_GET_ITEM(args[1], i), &ptrs[i]);
    Py_DECREF(t);
    if (!ok) return notServed();
  }
  PyObject *s = nullptr;
  if (args[3] == Py_None) {
    PyObject *device = PyObject_CallNoArgs(args[4]);
    if (device != nullptr) {
      s = PyObject_CallOneArg(args[5], device);
      Py_DECREF(device);
    }
  } else {
    s = PyObject_GetAttr(args[3], g_cudaStream);
  }
  const bool ok = s != nullptr && pointerOf(s, &stream);
  Py_XDECREF(s);
  if (!ok) return notServed();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = akg_hip_launch(static_cast<akg_hip_kernel_t *>(handle), ptrs, static_cast<int>(n), stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// launch_packed(handle, pointers, shapes, stream) -> (return code, address of the kernel that ran) or None
PyObject *launchPacked(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  if (nargs != 4 || !PyList_CheckExact(args[1]) || !PyList_CheckExact(args[2])) Py_RETURN_NONE;
  const Py_ssize_t n = PyList_GET_SIZE(args[1]);
  constexpr Py_ssize_t kMaxTensors = 64, kMaxRank = AKG_HIP_MAX_RANK;
  void *handle = nullptr, *stream = nullptr;
  void *ptrs[kMaxTensors];
  int64_t rows[kMaxTensors][1 + 2 * kMaxRank];   // [0, sizes, strides]
  const int64_t *lists[kMaxTensors];
  if (n > kMaxTensors || PyList_GET_SIZE(args[2]) != n || !pointerOf(args[0], &handle) || !pointerOf(args[3], &stream)) return notServed();
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject *shape = PyList_GET_ITEM(args[2], i);
    // torch.Size is a tuple; nothing below runs Python code, so the items stay
    if (!pointerOf(PyList_GET_ITEM(args[1], i), &ptrs[i]) || !(PyTuple_Check(shape) || PyList_CheckExact(shape))) return notServed();
    const Py_ssize_t rank = PySequence_Fast_GET_SIZE(shape);
    if (rank > kMaxRank) return notServed();
    int64_t *row = rows[i];
    for (Py_ssize_t d = 0; d < 1 + 2 * kMaxRank; ++d) row[d] = 0;
    for (Py_ssize_t d = 0; d < rank; ++d) {
      PyObject *extent = PySequence_Fast_GET_ITEM(shape, d);
      if (!PyLong_CheckExact(extent)) return notServed();
      row[1 + d] = PyLong_AsLongLong(extent);
      if (PyErr_Occurred()) return notServed();
    }
    uint64_t stride = 1;   // (wraps where a product of extents does not fit; such a shape fails the library's checks)
    for (Py_ssize_t d = rank; d-- > 0;) {
      row[1 + rank + d] = static_cast<int64_t>(stride);
      stride *= static_cast<uint64_t>(row[1 + d]);
    }
    lists[i] = row;
  }
  akg_hip_kernel_t *used = nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = akg_hip_dynamic_launch_packed(static_cast<akg_hip_dynamic_t *>(handle), ptrs, lists, static_cast<int>(n), stream, &used);
  Py_END_ALLOW_THREADS
  return Py_BuildValue("iN", rc, PyLong_FromVoidPtr(used));
}

PyMethodDef g_methods[] = {
    {"launch", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(launch)), METH_FASTCALL, "launch on device tensors"},
    {"launch_packed", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(launchPacked)), METH_FASTCALL, "dynamic-shape launch"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "akg_amd._launch", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__launch(void) {
  g_isCuda = PyUnicode_InternFromString("is_cuda");
  g_isContiguous = PyUnicode_InternFromString("is_contiguous");
  g_nbytes = PyUnicode_InternFromString("nbytes");
  g_dataPtr = PyUnicode_InternFromString("data_ptr");
  g_cudaStream = PyUnicode_InternFromString("cuda_stream");
  if (!g_isCuda || !g_isContiguous || !g_nbytes || !g_dataPtr || !g_cudaStream) return nullptr;
  return PyModule_Create(&g_module);
}
