"""Checks on lists of tensors that a hook makes every step, in native code (csrc/conef_host.cpp)."""
import importlib.util
import os
import struct
from functools import partial

from . import _lib

LIBPATH = os.path.join(os.path.dirname(_lib.LIBPATH), "libconef_host.so")

_module = None


def load():
    """Loads the helper module (once).  Raises if it is not built."""
    global _module
    if _module is None:
        if not os.path.exists(LIBPATH):
            raise _lib.ConefLibraryError("libconef_host.so is not built (expected at %s); run `python -m conef_amd.build`."
                                         % LIBPATH)
        spec = importlib.util.spec_from_file_location("libconef_host", LIBPATH)
        module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
        _module = module
    return _module


def _words(numbers):
    return struct.pack("=%dq" % len(numbers), *numbers)


def same_shapes(tensors):
    """A function of a list of tensors: whether it has the shapes of this one, in order."""
    return partial(load().same_shapes, _words([w for t in tensors for w in (t.dim(), *t.shape)]))


def same_places(tensors):
    """A function of a list of tensors: whether their memory starts where that of these does."""
    return partial(load().same_places, _words([t.data_ptr() for t in tensors]))


def same_sketches(sketches, moves):
    """A function of a list of sketches: whether they are these very objects, with the plans they have now, and
    with their cells where they are now if they are updated in place (``moves[i]``: sketch i swaps two
    buffers, its cells may be anywhere)."""
    sketches = list(sketches)
    places = [0 if m else s.cs.data_ptr() for s, m in zip(sketches, moves)]
    return partial(load().same_sketches, _words(places), sketches, [s._plan for s in sketches])
