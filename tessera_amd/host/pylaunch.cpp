// The Python side of one launch, as a CPython extension: KernelLaunch's attributes to the argument
// arrays of qmm_launch.  backend.py does everything else over ctypes; this call is the one that a
// decode step makes for every kernel, and building the arrays through ctypes objects took more of the
// processor's time (3.3 us of 5.6 a launch) than the launch itself.
//
// launch(entry, kernel, launch, stream) -> status: `entry` is the address of qmm_launch or
// qmm_launch_static, `kernel` the handle, `launch` a KernelLaunch (its buffers have Handle() and
// Size()).  Numbers wrap as C integers do, the interpreter lock is released during the call.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstddef>
#include <cstdint>

#include "../../include/tessera_qmm.h"

namespace {

using Entry = qmm_status (*)(qmm_kernel, const uint32_t*, const uint32_t*, void* const*, const size_t*, size_t, const uint64_t*,
                             size_t, void*);

PyObject *s_grid[3], *s_block[3], *s_buffers, *s_scalars, *s_handle, *s_size;

// int(value) modulo 2^64; false with a Python error set.
bool whole(PyObject* value, uint64_t* out) {
  if (PyLong_Check(value)) {
    *out = PyLong_AsUnsignedLongLongMask(value);
  } else {
    PyObject* number = PyNumber_Long(value);
    if (number == nullptr) return false;
    *out = PyLong_AsUnsignedLongLongMask(number);
    Py_DECREF(number);
  }
  return !(*out == ~0ull && PyErr_Occurred());
}

bool attribute(PyObject* owner, PyObject* name, uint64_t* out) {
  PyObject* value = PyObject_GetAttr(owner, name);
  if (value == nullptr) return false;
  const bool ok = whole(value, out);
  Py_DECREF(value);
  return ok;
}

bool method(PyObject* owner, PyObject* name, uint64_t* out) {
  PyObject* value = PyObject_CallMethodNoArgs(owner, name);
  if (value == nullptr) return false;
  bool ok = true;
  if (value == Py_None) {
    *out = 0;
  } else {
    ok = whole(value, out);
  }
  Py_DECREF(value);
  return ok;
}

// The elements that owner.name has now, up to N of them held, and their whole number: what is called on them may run
// Python code, and that (or another thread meanwhile) may change the list.  (A tuple of them costs 25 ns more.)
template <int N>
struct Snapshot {
  PyObject* item[N];
  Py_ssize_t held = 0, count = -1;   // count < 0: a Python error is set

  Snapshot(PyObject* owner, PyObject* name) {
    PyObject* list = PyObject_GetAttr(owner, name);
    if (list == nullptr) return;
    PyObject* items = PySequence_Fast(list, "buffers and scalars must be sequences");
    Py_DECREF(list);
    if (items == nullptr) return;
    count = PySequence_Fast_GET_SIZE(items);
    for (; held < count && held < N; ++held) {
      item[held] = PySequence_Fast_GET_ITEM(items, held);
      Py_INCREF(item[held]);
    }
    Py_DECREF(items);
  }
  ~Snapshot() {
    for (Py_ssize_t i = 0; i < held; ++i) Py_DECREF(item[i]);
  }
  Snapshot(const Snapshot&) = delete;
  Snapshot& operator=(const Snapshot&) = delete;
};

PyObject* launch(PyObject*, PyObject* const* args, Py_ssize_t count) {
  if (count != 4) {
    PyErr_SetString(PyExc_TypeError, "launch(entry, kernel, launch, stream)");
    return nullptr;
  }
  uint64_t entry, kernel, stream, v;
  if (!whole(args[0], &entry) || !whole(args[1], &kernel) || !whole(args[3], &stream)) return nullptr;
  uint32_t grid[3], block[3];
  for (int i = 0; i < 3; ++i) {
    if (!attribute(args[2], s_grid[i], &v)) return nullptr;
    grid[i] = static_cast<uint32_t>(v);
    if (!attribute(args[2], s_block[i], &v)) return nullptr;
    block[i] = static_cast<uint32_t>(v);
  }
  // More than the limits: the count is passed on, and qmm_launch refuses it before it reads an entry.
  void* handles[QMM_MAX_BOUND_BUFFERS];
  size_t sizes[QMM_MAX_BOUND_BUFFERS];
  uint64_t scalars[QMM_MAX_SCALARS];
  const Snapshot<QMM_MAX_BOUND_BUFFERS> buffer(args[2], s_buffers);
  if (buffer.count < 0) return nullptr;
  for (Py_ssize_t i = 0; i < buffer.held; ++i) {
    if (!method(buffer.item[i], s_handle, &v)) return nullptr;
    handles[i] = reinterpret_cast<void*>(v);
    if (!method(buffer.item[i], s_size, &v)) return nullptr;
    sizes[i] = static_cast<size_t>(v);
  }
  const Snapshot<QMM_MAX_SCALARS> scalar(args[2], s_scalars);
  if (scalar.count < 0) return nullptr;
  for (Py_ssize_t i = 0; i < scalar.held; ++i) {
    if (!whole(scalar.item[i], &scalars[i])) return nullptr;
  }
  qmm_status status;
  Py_BEGIN_ALLOW_THREADS
  status = reinterpret_cast<Entry>(entry)(static_cast<qmm_kernel>(kernel), grid, block, handles, sizes, static_cast<size_t>(buffer.count),
                                          scalars, static_cast<size_t>(scalar.count), reinterpret_cast<void*>(stream));
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(status);
}

PyMethodDef kMethods[] = {
    {"launch", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(launch)), METH_FASTCALL,
     "launch(entry, kernel, launch, stream) -> status"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "One qmm_launch from a KernelLaunch.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
  const char* names[] = {"grid_x", "grid_y", "grid_z", "block_x", "block_y", "block_z", "buffers", "scalars", "Handle", "Size"};
  PyObject** slots[] = {&s_grid[0], &s_grid[1], &s_grid[2], &s_block[0], &s_block[1], &s_block[2],
                        &s_buffers, &s_scalars, &s_handle, &s_size};
  for (size_t i = 0; i < sizeof(slots) / sizeof(slots[0]); ++i) {
    *slots[i] = PyUnicode_InternFromString(names[i]);
    if (*slots[i] == nullptr) return nullptr;
  }
  return PyModule_Create(&kModule);
}
