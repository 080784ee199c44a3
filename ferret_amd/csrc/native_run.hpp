// One C-ABI call of the native call path (native.cpp), its return code sorted
// into done, left to Python, and raised.  Needs nothing but Python.h, so that a
// CPU test compiles it.
#pragma once
#include <Python.h>

namespace ferret {
namespace native {

// Raises ferret_amd.lib.FerretError for a code of `entry`.
inline void raise_code(const char* entry, int rc) {
  PyObject* lib = PyImport_ImportModule("ferret_amd.lib");
  PyObject* none = lib != nullptr ? PyObject_CallMethod(lib, "check", "si", entry, rc) : nullptr;
  Py_XDECREF(none);
  Py_XDECREF(lib);
}

// The interpreter lock given up for a scope.  Taken back also where a C++
// exception leaves it: the function's handler sets a Python error, which needs it.
class Unlocked {
 public:
  Unlocked() : state_(PyEval_SaveThread()) {}
  ~Unlocked() { PyEval_RestoreThread(state_); }
  Unlocked(const Unlocked&) = delete;
  Unlocked& operator=(const Unlocked&) = delete;

 private:
  PyThreadState* state_;
};

// f() is the C call of `entry`, made without the interpreter lock (as ctypes
// makes it).  True where it returned 0.  A negative code was returned before
// anything was launched: the Python path makes the call again and names the
// error.  A positive one is the HIP runtime's: reading it has cleared it there,
// and kernels of the operator may be on the stream already, so that a second call
// would hide the error and enqueue them twice.  It is raised here.
template <typename F>
bool run(const char* entry, F&& f) {
  int rc;
  {
    const Unlocked unlocked;
    rc = f();
  }
  if (rc > 0) raise_code(entry, rc);
  return rc == 0;
}

// What a function returns after run() gave false: null where an error was raised,
// else None, which leaves the call to the Python path.
inline PyObject* declined() {
  if (PyErr_Occurred() != nullptr) return nullptr;
  Py_RETURN_NONE;
}

}  // namespace native
}  // namespace ferret
