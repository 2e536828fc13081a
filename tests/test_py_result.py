"""Return values of the operator layer's native calls when Python runs out of memory while they are built: an exception,
and every object made so far is given up (CPU; the header is compiled with constructors that fail on demand)."""
import importlib.util
import os
import subprocess
import sys
import sysconfig

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <Python.h>
static int g_left = -1;                       /* constructors that still succeed; -1: all of them */
static bool fails() { if (g_left == 0) { PyErr_NoMemory(); return true; } if (g_left > 0) --g_left; return false; }
static PyObject *new_tuple(Py_ssize_t n) { return fails() ? nullptr : PyTuple_New(n); }
static PyObject *new_list(Py_ssize_t n) { return fails() ? nullptr : PyList_New(n); }
static PyObject *new_long(long long v) { return fails() ? nullptr : PyLong_FromLongLong(v); }
#define PyTuple_New new_tuple
#define PyList_New new_list
#define PyLong_FromLongLong new_long
#include "zbal_py_result.h"

static Owned again(PyObject *o) { if (fails()) throw PyFail{}; Py_INCREF(o); return Owned(o); }

/* (object, constructors that succeed) -> (object, object, [2, 5]) */
static PyObject *build(PyObject *, PyObject *const *args, Py_ssize_t)
{
    g_left = (int)PyLong_AsLong(args[1]);
    try {
        return tuple_of(again(args[0]), again(args[0]), list_of({2, 3}, true));
    } catch (const PyFail &) {
        return nullptr;
    }
}
static PyMethodDef methods[] = {{"build", (PyCFunction)(void (*)(void))build, METH_FASTCALL, nullptr}, {nullptr, nullptr, 0, nullptr}};
static PyModuleDef module = {PyModuleDef_HEAD_INIT, "py_result_test", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};
PyMODINIT_FUNC PyInit_py_result_test() { return PyModule_Create(&module); }
"""


@pytest.fixture(scope="module")
def build(tmp_path_factory):
    d = tmp_path_factory.mktemp("py_result")
    (d / "t.cpp").write_text(SOURCE)
    so = str(d / "py_result_test.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I" + sysconfig.get_paths()["include"],
                           "-I" + os.path.join(ROOT, "memfabric_hybrid_amd", "csrc", "torch"), str(d / "t.cpp"), "-o", so])
    spec = importlib.util.spec_from_file_location("py_result_test", so)
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module.build


def test_a_result_that_cannot_be_built_leaves_nothing_behind(build):
    thing = object()
    before = sys.getrefcount(thing)
    whole = build(thing, -1)
    assert whole == (thing, thing, [2, 5])
    del whole
    for succeed in range(6):                  # two references, the list, its two integers, the tuple
        with pytest.raises(MemoryError):
            build(thing, succeed)
        assert sys.getrefcount(thing) == before, succeed
    assert build(thing, 6) == (thing, thing, [2, 5])
    assert sys.getrefcount(thing) == before
