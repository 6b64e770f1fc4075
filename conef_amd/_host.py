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
        for fn in (lib.conef_host_same_shapes, lib.conef_host_same_places):
            fn.argtypes, fn.restype = [ctypes.py_object, ctypes.c_void_p, ctypes.c_int64], ctypes.c_int
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
    """Where the memory of a list of tensors, or of sketches (their cells), starts."""
    __slots__ = ("words", "at", "n", "check")

    def __init__(self, holders):
        words = [getattr(h, "cs", h).data_ptr() for h in holders]
        self.n = len(words)
        self.words = (ctypes.c_int64 * self.n)(*words)
        self.at = ctypes.addressof(self.words)
        self.check = load().conef_host_same_places

    def same(self, holders):
        return bool(self.check(holders, self.at, self.n))
