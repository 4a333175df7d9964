// A module around csrc_torch/unlocked.h for tests/test_native_calls.py.
#include "unlocked.h"

#include <stdexcept>

namespace {

int work(int x, int fail) {
  if (fail) throw std::runtime_error("thrown without the lock");
  return PyGILState_Check() ? -1 : x + 1;      // (-1: the lock was still held)
}

int read(int fail) {
  if (fail) throw std::runtime_error(PyGILState_Check() ? "thrown with the lock" : "lock lost");
  return 41;
}

// call(where): where 0 nothing throws, 1 the call does, 2 reading its argument does
PyObject* call(PyObject*, PyObject* o) {
  const long where = PyLong_AsLong(o);
  try {
    return PyLong_FromLong(dq8::call_unlocked(work, read(where == 2), where == 1 ? 1 : 0));
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

PyMethodDef kMethods[] = {{"call", call, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "unlocked_module", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_unlocked_module(void) { return PyModule_Create(&kModule); }
