"""ctypes binding of libpgrav.so (the C ABI declared in include/pgrav.h).

The shared library is built in-tree by ahotsph-2hot-apps_amd/build.py.  There is
no fallback: if the library is missing, every entry point raises.
"""
import ctypes
import os

import numpy as np

PKG = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
# PGRAV_LIBRARY selects another build of the same ABI (e.g. a variant built
# with build.py --out); the default is the in-tree library
LIB_PATH = os.environ.get("PGRAV_LIBRARY") or os.path.join(PKG, "libpgrav.so")


class PgravError(RuntimeError):
    pass


_lib = None

_f32p = np.ctypeslib.ndpointer(np.float32, flags="C_CONTIGUOUS")
_vp = ctypes.c_void_p
_i = ctypes.c_int
_i64 = ctypes.c_int64
_f = ctypes.c_float
_d = ctypes.c_double
_cp = ctypes.c_char_p


class Segment(ctypes.Structure):
    """nln/segment.h:16-19"""
    _fields_ = [("base", ctypes.c_uint), ("length", ctypes.c_uint)]


# name -> (restype, argtypes); every symbol of include/pgrav.h
SIGNATURES = {
    "CUDA_Init": (None, [_vp]),
    "CUDA_Finalize": (None, []),
    "vecwidthCUDA": (_i, []),
    "qallocCUDA": (_i, [_vp]),
    "WalkInitSrcCUDA": (None, [_vp, _i, _i64]),
    "WalkTerminateSrcCUDA": (None, []),
    "WalkInitSinkCUDA": (None, [_vp, _i, _i64]),
    "WalkTerminateSinkCUDA": (None, [_vp, _i, _i64]),
    "grav_mn_CUDA": (None, [_cp, _vp, _vp, _i, _i, _vp, _i, _i, _f, _vp, _i]),
    "grav_mns_CUDA": (None, [_cp, _i, _i, _vp, _i, _i, _f, _f, _vp, _i]),
    "grav_mnss_CUDA": (None, [_cp, _i, _i, _vp, _vp, _i, _vp, _i, _i, _vp, _f, _f, _vp, _i]),
    "grav_qns_CUDA": (None, [_cp, _i, _i, _vp, _i, _i]),
    "grav_qnss_CUDA": (None, [_cp, _i, _i, _vp, _vp, _i, _i]),
    "pinteractCUDA": (None, [_vp, _vp, _i, _i, _vp, _i, _i, _i]),
    "pgrav_mn_host": (_i, [_i, _vp, _vp, _i, _i, _vp, _i, _i, _i, _f]),
    "pgrav_set_error_mode": (_i, [_i]),
    "pgrav_last_error": (_cp, []),
    "pgrav_clear_error": (None, []),
    "pgrav_set_quad_phi_sign": (None, [_i]),
    "pgrav_synchronize": (_i, []),
    "pgrav_set_dropin_deferral": (_i, [_i]),
}


def lib():
    """Loads libpgrav.so once; raises PgravError if it has not been built."""
    global _lib
    if _lib is None:
        if not os.path.exists(LIB_PATH):
            raise PgravError(LIB_PATH + " is not built: run "
                             "python ahotsph-2hot-apps_amd/build.py (no CPU fallback exists)")
        L = ctypes.CDLL(LIB_PATH)
        for name, (res, args) in SIGNATURES.items():
            fn = getattr(L, name)
            fn.restype = res
            fn.argtypes = args
        for name, (res, args) in _EXTRA.items():
            if hasattr(L, name):
                fn = getattr(L, name)
                fn.restype = res
                fn.argtypes = args
        L.pgrav_set_error_mode(1)  # record errors; raise them from Python
        _lib = L
    return _lib


_EXTRA = {}


def register(signatures):
    """Adds signatures for later parts of the ABI (batched path)."""
    _EXTRA.update(signatures)
    SIGNATURES.update(signatures)
    if _lib is not None:
        for name, (res, args) in signatures.items():
            fn = getattr(_lib, name)
            fn.restype = res
            fn.argtypes = args


def check():
    """Raises the error recorded by the last call, if any."""
    L = lib()
    msg = L.pgrav_last_error()
    if msg is not None:
        L.pgrav_clear_error()
        raise PgravError(msg.decode())


def ptr(a):
    """Raw pointer of a numpy array (or None).  Through the buffer protocol: numpy's own
    a.ctypes.data costs 2.5 us, more than most drop-in calls; it serves the arrays whose
    buffer ctypes does not take (read-only, empty, not C-contiguous) and refuses what is
    no array, which may well have a buffer."""
    if a is None:
        return None
    if isinstance(a, np.ndarray):
        try:
            return ctypes.c_void_p(ctypes.addressof(ctypes.c_char.from_buffer(a)))
        except (TypeError, ValueError, BufferError):
            pass
    return ctypes.c_void_p(a.ctypes.data)
