/*
 * Return values of the native calls: Python objects that are given up again if a later one cannot be made.
 */
#ifndef ZBAL_PY_RESULT_H_
#define ZBAL_PY_RESULT_H_

#include <Python.h>

#include <cstdint>
#include <memory>
#include <vector>

namespace {

/* a Python exception is set */
struct PyFail {};

struct Drop {
    void operator()(PyObject *o) const { Py_XDECREF(o); }
};
using Owned = std::unique_ptr<PyObject, Drop>;

inline Owned checked(PyObject *o)
{
    if (o == nullptr) throw PyFail{};
    return Owned(o);
}

template <typename... T> PyObject *tuple_of(T... items)
{
    Owned all[] = {std::move(items)...};
    Owned r = checked(PyTuple_New(sizeof...(items)));
    for (size_t i = 0; i < sizeof...(items); ++i) PyTuple_SET_ITEM(r.get(), (Py_ssize_t)i, all[i].release());
    return r.release();
}

/* the counts, or their running sums, as a list of integers */
inline Owned list_of(const std::vector<int64_t> &counts, bool running)
{
    Owned r = checked(PyList_New((Py_ssize_t)counts.size()));
    int64_t run = 0;
    for (size_t e = 0; e < counts.size(); ++e) {
        run = running ? run + counts[e] : counts[e];
        PyList_SET_ITEM(r.get(), (Py_ssize_t)e, checked(PyLong_FromLongLong(run)).release());
    }
    return r;
}

} // namespace

#endif /* ZBAL_PY_RESULT_H_ */
