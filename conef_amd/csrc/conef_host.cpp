// Host-side checks a hook makes on every step before it relies on the tables it keeps for a bucket:
// has every gradient the shape it had, do the error tensors and sketches lie where they lay?
//
// The answers are a walk over a Python list.  In Python that is 0.15 us a tensor (a torch.Size object
// each): 9 us for the 59 gradients of a ResNet-20, whose whole step is 21 us.  Here the sizes are read
// where they are: 0.8 us for the 59 on the same machine.  Plain C entry points, called through
// ctypes.PyDLL (the GIL stays held); anything unexpected answers "no", and the caller then builds its
// tables anew, which raises whatever there is to raise.
#include <torch/csrc/autograd/python_variable.h>

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

// 1 if the memory of holders[i] - a tensor, or an object whose attribute `cs` is one - starts at places[i]
// for every i below n, and there are n of them.
int conef_host_same_places(PyObject* holders, const int64_t* places, int64_t n)
{
    static PyObject* const cells = PyUnicode_InternFromString("cs");
    PyObject* seq = PySequence_Fast(holders, "");
    if (!seq) {
        PyErr_Clear();
        return 0;
    }
    int same = cells && PySequence_Fast_GET_SIZE(seq) == (Py_ssize_t)n;
    for (int64_t i = 0; i < n && same; ++i) {
        // (the exact type first: asking a sketch whether it is a tensor goes through Python)
        PyObject* o = PySequence_Fast_GET_ITEM(seq, i);
        PyObject* inner = THPVariable_CheckExact(o) ? nullptr : PyObject_GetAttr(o, cells);
        if (inner) {
            o = inner;
        } else {
            PyErr_Clear();
            Py_INCREF(o);
        }
        try {
            same = THPVariable_Check(o) && (int64_t)(intptr_t)THPVariable_Unpack(o).data_ptr() == places[i];
        } catch (...) {
            same = 0;
        }
        Py_DECREF(o);
    }
    Py_DECREF(seq);
    if (!same) PyErr_Clear();
    return same;
}

}  // extern "C"
