"""The renderer's host code built for the CPU over a stand-in HIP runtime
(tests/hostabi): a Renderer whose device memory is host memory with a limit, and
whose ray queries run on the CPU. Test infrastructure; the product never loads it."""
import ctypes as C
import os
import subprocess

from glslpt import _capi as api
from glslpt.renderer import Renderer

ROOT = os.path.dirname(os.path.abspath(__file__))
PATH = os.path.join(ROOT, "hostabi", "_build", "libhostabi.so")

_lib = None


def lib():
    global _lib
    if _lib is None:
        subprocess.check_call(["make", "-s", "-C", os.path.join(ROOT, "hostabi")])
        _lib = C.CDLL(PATH)
        for fn, args in api._HIP_SIGS.items():
            if hasattr(_lib, fn):
                getattr(_lib, fn).argtypes = args
                getattr(_lib, fn).restype = C.c_int
        _lib.pt_last_error.argtypes = [C.c_void_p]
        _lib.pt_last_error.restype = C.c_char_p
        for fn in ("fake_device_used", "fake_device_peak", "fake_pinned"):
            getattr(_lib, fn).restype = C.c_size_t
        _lib.fake_device_limit.argtypes = [C.c_size_t]
        _lib.fake_device_limit.restype = None
    return _lib


class HostRenderer(Renderer):
    def __init__(self):
        self._lib = lib()
        h = C.c_void_p()
        assert self._lib.pt_create(0, C.byref(h)) == api.PT_OK
        self._h = h
        self.width = self.height = 0
