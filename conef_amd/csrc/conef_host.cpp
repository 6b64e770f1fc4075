// Host-side checks a hook makes on every step before it relies on the tables it keeps for a bucket:
// has every gradient the shape it had, do the error tensors and sketches lie where they lay?
//
// The answers are a walk over a Python list.  In Python that is 0.15 us a tensor (a torch.Size object
// each): 9 us for the 59 gradients of a ResNet-20, whose whole step is 21 us.  Here the sizes are read
// where they are: 0.8 us for the 59 on the same machine.  Plain C entry points, called through
// ctypes.PyDLL (the GIL stays held); anything unexpected answers "no", and the caller then builds its
// tables anew, which raises whatever there is to raise.
#include <torch/csrc/autograd/python_variable.h>

namespace {

bool starts_at(PyObject* tensor, int64_t place)
{
    if (!THPVariable_Check(tensor)) return false;
    try {
        return (int64_t)(intptr_t)THPVariable_Unpack(tensor).data_ptr() == place;
    } catch (...) {
        return false;
    }
}

}  // namespace

extern "C" {

// 1 if `tensors` (a list or tuple) holds tensors of the shapes in want[0 .. n): per tensor the number of
// dimensions, then the dimensions.
int conef_host_same_shapes(PyObject* tensors, const int64_t* want, int64_t n)
{
    PyObject* seq = PySequence_Fast(tensors, "");
    if (!seq) {
        PyErr_Clear();
        return 0;
    }
    const int64_t* end = want + n;
    int same = 1;
    try {
        const Py_ssize_t count = PySequence_Fast_GET_SIZE(seq);
        for (Py_ssize_t i = 0; i < count && same; ++i) {
            PyObject* o = PySequence_Fast_GET_ITEM(seq, i);
            if (!THPVariable_Check(o)) {
                same = 0;
                break;
            }
            const auto sizes = THPVariable_Unpack(o).sizes();
            if (end - want < 1 + (int64_t)sizes.size() || *want++ != (int64_t)sizes.size()) {
                same = 0;
                break;
            }
            for (const int64_t d : sizes) same &= *want++ == d;
        }
        same &= want == end;
    } catch (...) {
        same = 0;
    }
    Py_DECREF(seq);
    return same;
}

// 1 if the memory of tensors[i] starts at places[i] for every i below n, and there are n of them.
int conef_host_same_places(PyObject* tensors, const int64_t* places, int64_t n)
{
    PyObject* seq = PySequence_Fast(tensors, "");
    if (!seq) {
        PyErr_Clear();
        return 0;
    }
    int same = PySequence_Fast_GET_SIZE(seq) == (Py_ssize_t)n;
    for (int64_t i = 0; i < n && same; ++i) same = starts_at(PySequence_Fast_GET_ITEM(seq, i), places[i]);
    Py_DECREF(seq);
    return same;
}

// 1 if `sketches` holds the very objects of the list `known`, each with the object of the list `plans` as its
// attribute _plan and its cells (attribute cs, a tensor) at places[i], where places[i] is not 0.
int conef_host_same_sketches(PyObject* sketches, PyObject* known, PyObject* plans, const int64_t* places, int64_t n)
{
    static PyObject* const cells = PyUnicode_InternFromString("cs");
    static PyObject* const plan = PyUnicode_InternFromString("_plan");
    PyObject* seq = PySequence_Fast(sketches, "");
    if (!seq) {
        PyErr_Clear();
        return 0;
    }
    int same = cells && plan && PyList_Check(known) && PyList_Check(plans) && PySequence_Fast_GET_SIZE(seq) == (Py_ssize_t)n &&
               PyList_GET_SIZE(known) == (Py_ssize_t)n && PyList_GET_SIZE(plans) == (Py_ssize_t)n;
    for (int64_t i = 0; i < n && same; ++i) {
        PyObject* o = PySequence_Fast_GET_ITEM(seq, i);
        same = o == PyList_GET_ITEM(known, i);
        if (!same) break;
        PyObject* p = PyObject_GetAttr(o, plan);
        same = p == PyList_GET_ITEM(plans, i);
        Py_XDECREF(p);
        if (!same || places[i] == 0) continue;
        PyObject* t = PyObject_GetAttr(o, cells);
        same = t && starts_at(t, places[i]);
        Py_XDECREF(t);
    }
    Py_DECREF(seq);
    if (!same) PyErr_Clear();
    return same;
}

}  // extern "C"
