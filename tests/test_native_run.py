"""Return codes of the native call path (ferret_amd/csrc/native_run.hpp), on the CPU: a small module made of that
header, with a C call that counts its runs and gives any code."""
import importlib.util
import os
import shutil
import subprocess
import sysconfig

import pytest

from ferret_amd import lib

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ferret_amd", "csrc")

MODULE = r"""
#include "native_run.hpp"
#include <stdexcept>
using namespace ferret::native;
static int calls = 0;
static PyObject* call(PyObject*, PyObject* code) {
  const int rc = (int)PyLong_AsLong(code);
  if (!run("ferret_entry", [&] { ++calls; return rc; })) return declined();
  return PyUnicode_FromString("done");
}
static PyObject* fail(PyObject*, PyObject*) {
  try {
    run("ferret_entry", []() -> int { throw std::runtime_error("no storage"); });
  } catch (const std::exception& e) {  // as the functions of native.cpp do
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
  Py_RETURN_NONE;
}
static PyObject* count(PyObject*, PyObject*) { return PyLong_FromLong(calls); }
static PyMethodDef kMethods[] = {{"call", call, METH_O, nullptr}, {"fail", fail, METH_NOARGS, nullptr},
                                 {"count", count, METH_NOARGS, nullptr},
                                 {nullptr, nullptr, 0, nullptr}};
static PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "run_probe", "", -1, kMethods, nullptr, nullptr, nullptr, nullptr};
PyMODINIT_FUNC PyInit_run_probe(void) { return PyModule_Create(&kModule); }
"""


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("run_probe")
    src, so = d / "run_probe.cpp", d / "run_probe.so"
    src.write_text(MODULE)
    subprocess.run([gxx, "-std=c++17", "-O1", "-fPIC", "-shared", f"-I{CSRC}", f"-I{sysconfig.get_paths()['include']}",
                    str(src), "-o", str(so)], check=True)
    spec = importlib.util.spec_from_file_location("run_probe", so)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


class _Library:
    @staticmethod
    def ferret_error_string(code):
        return b"text %d" % code


def test_hip_errors_are_raised_and_rejected_arguments_left_to_python(probe, monkeypatch):
    monkeypatch.setattr(lib, "load", _Library)
    before = probe.count()
    assert probe.call(0) == "done"
    assert probe.call(-2) is None
    with pytest.raises(lib.FerretError, match="ferret_entry failed with code 719: text 719") as e:
        probe.call(719)
    assert e.value.code == 719
    assert probe.count() == before + 3      # each code came from one call


def test_a_cpp_exception_leaves_the_interpreter_lock_held(probe):
    """A pointer taken inside the call can throw (a tensor without storage, a copy-on-write one out of memory)."""
    with pytest.raises(RuntimeError, match="no storage"):
        probe.fail()
