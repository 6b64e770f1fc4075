// Host-side checks a hook makes on every step before it relies on the tables it keeps for a bucket:
// has every gradient the shape it had, do the error tensors and sketches lie where they lay?
//
// The answers are a walk over a Python list.  In Python that is 0.15 us a tensor (a torch.Size object
// each): 9 us for the 59 gradients of a ResNet-20, whose whole step is 21 us.  Here the sizes are read
// where they are.  A small CPython module; `words` is a bytes object of 64-bit numbers the caller packed.
// Anything unexpected answers False, and the caller then builds its tables anew, which raises whatever
// there is to raise.
#include <torch/csrc/autograd/python_variable.h>

namespace {

// the 64-bit numbers of a bytes object
struct Words {
    const char* at = nullptr;
    Py_ssize_t n = -1;
    explicit Words(PyObject* o)
    {
        if (PyBytes_Check(o)) {
            at = PyBytes_AS_STRING(o);
            n = PyBytes_GET_SIZE(o) / 8;
        }
    }
    int64_t operator[](Py_ssize_t i) const
    {
        int64_t v;
        memcpy(&v, at + 8 * i, 8);
        return v;
    }
};

// a list or tuple (made one where it is neither), or null with no error left
PyObject* sequence(PyObject* o)
{
    PyObject* seq = PySequence_Fast(o, "");
    if (!seq) PyErr_Clear();
    return seq;
}

bool shapes_are(PyObject* seq, const Words& want)
{
    try {
        const Py_ssize_t count = PySequence_Fast_GET_SIZE(seq);
        Py_ssize_t w = 0;
        for (Py_ssize_t i = 0; i < count; ++i) {
            PyObject* o = PySequence_Fast_GET_ITEM(seq, i);
            if (!THPVariable_Check(o)) return false;
            const auto sizes = THPVariable_Unpack(o).sizes();
            if (want.n - w < 1 + (Py_ssize_t)sizes.size() || want[w++] != (int64_t)sizes.size()) return false;
            for (const int64_t d : sizes)
                if (want[w++] != d) return false;
        }
        return w == want.n;
    } catch (...) {
        return false;
    }
}

bool starts_at(PyObject* tensor, int64_t place)
{
    if (!THPVariable_Check(tensor)) return false;
    try {
        return (int64_t)(intptr_t)THPVariable_Unpack(tensor).data_ptr() == place;
    } catch (...) {
        return false;
    }
}

// same_shapes(words, tensors): the tensors have the shapes in `words` - per tensor the number of dimensions, then
// the dimensions
PyObject* same_shapes(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    if (nargs != 2) return PyErr_Format(PyExc_TypeError, "same_shapes(words, tensors)");
    const Words want(args[0]);
    PyObject* seq = sequence(args[1]);
    const bool same = seq && want.n >= 0 && shapes_are(seq, want);
    Py_XDECREF(seq);
    return PyBool_FromLong(same);
}

// same_places(words, tensors): as many tensors as words, the memory of tensor i starts at word i
PyObject* same_places(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    if (nargs != 2) return PyErr_Format(PyExc_TypeError, "same_places(words, tensors)");
    const Words places(args[0]);
    PyObject* seq = sequence(args[1]);
    bool same = seq && PySequence_Fast_GET_SIZE(seq) == places.n;
    for (Py_ssize_t i = 0; same && i < places.n; ++i) same = starts_at(PySequence_Fast_GET_ITEM(seq, i), places[i]);
    Py_XDECREF(seq);
    return PyBool_FromLong(same);
}

// same_sketches(words, known, plans, sketches): the very objects of the list `known`, each with the object of the
// list `plans` as its attribute _plan and its cells (attribute cs, a tensor) at word i, where that is not 0
PyObject* same_sketches(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    static PyObject* const cells = PyUnicode_InternFromString("cs");
    static PyObject* const plan = PyUnicode_InternFromString("_plan");
    if (nargs != 4) return PyErr_Format(PyExc_TypeError, "same_sketches(words, known, plans, sketches)");
    const Words places(args[0]);
    PyObject *known = args[1], *plans = args[2];
    PyObject* seq = sequence(args[3]);
    bool same = seq && cells && plan && PyList_Check(known) && PyList_Check(plans) && PySequence_Fast_GET_SIZE(seq) == places.n &&
                PyList_GET_SIZE(known) == places.n && PyList_GET_SIZE(plans) == places.n;
    for (Py_ssize_t i = 0; same && i < places.n; ++i) {
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
    Py_XDECREF(seq);
    if (!same) PyErr_Clear();
    return PyBool_FromLong(same);
}

PyMethodDef methods[] = {
    {"same_shapes", (PyCFunction)(void (*)(void))same_shapes, METH_FASTCALL, nullptr},
    {"same_places", (PyCFunction)(void (*)(void))same_places, METH_FASTCALL, nullptr},
    {"same_sketches", (PyCFunction)(void (*)(void))same_sketches, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "libconef_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_libconef_host(void) { return PyModule_Create(&module); }
