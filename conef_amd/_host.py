"""Checks on lists of tensors that a hook makes every step, in native code (csrc/conef_host.cpp)."""
import ctypes
import os

from . import _lib

LIBPATH = os.path.join(os.path.dirname(_lib.LIBPATH), "libconef_host.so")

_handle = None


def load():
    """Loads the helper library (once).  Raises if it is not built."""
    global _handle
    if _handle is None:
        if not os.path.exists(LIBPATH):
            raise _lib.ConefLibraryError("libconef_host.so is not built (expected at %s); run `python -m conef_amd.build`."
                                         % LIBPATH)
        lib = ctypes.PyDLL(LIBPATH)
        objects, words, count = ctypes.py_object, ctypes.c_void_p, ctypes.c_int64
        lib.conef_host_same_shapes.argtypes = lib.conef_host_same_places.argtypes = [objects, words, count]
        lib.conef_host_same_sketches.argtypes = [objects, objects, objects, words, count]
        for fn in (lib.conef_host_same_shapes, lib.conef_host_same_places, lib.conef_host_same_sketches):
            fn.restype = ctypes.c_int
        _handle = lib
    return _handle


class Shapes:
    """The shapes of a list of tensors, in order; ``same(tensors)`` compares another list's."""
    __slots__ = ("words", "at", "n", "check")

    def __init__(self, tensors):
        words = [w for t in tensors for w in (t.dim(), *t.shape)]
        self.n = len(words)
        self.words = (ctypes.c_int64 * self.n)(*words)
        self.at = ctypes.addressof(self.words)
        self.check = load().conef_host_same_shapes

    def same(self, tensors):
        return bool(self.check(tensors, self.at, self.n))


class Places:
    """Where the memory of a list of tensors starts."""
    __slots__ = ("words", "at", "n", "check")

    def __init__(self, tensors):
        self.n = len(tensors)
        self.words = (ctypes.c_int64 * self.n)(*[t.data_ptr() for t in tensors])
        self.at = ctypes.addressof(self.words)
        self.check = load().conef_host_same_places

    def same(self, tensors):
        return bool(self.check(tensors, self.at, self.n))


class Sketches:
    """A list of sketches: the objects, their plans, and where the cells of those start that are updated in
    place (``moves[i]``: sketch i swaps two buffers, its cells may be anywhere)."""
    __slots__ = ("known", "plans", "words", "at", "n", "check")

    def __init__(self, sketches, moves):
        self.known, self.plans, self.n = list(sketches), [s._plan for s in sketches], len(sketches)
        self.words = (ctypes.c_int64 * self.n)(*[0 if m else s.cs.data_ptr() for s, m in zip(sketches, moves)])
        self.at = ctypes.addressof(self.words)
        self.check = load().conef_host_same_sketches

    def same(self, sketches):
        return bool(self.check(sketches, self.known, self.plans, self.at, self.n))
