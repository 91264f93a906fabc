"""The product of gemm_residue.hip called directly, for the tests: the library's C++ symbols by
ctypes, with a workspace and a flag of the caller's."""
import ctypes
import functools
import subprocess

import numpy as np

import mcnla_amd as mc
from mcnla_amd import _lib


class ResidueArgs(ctypes.Structure):
    """mcnla::ResidueArgs (kernels.hpp)."""
    _fields_ = [("M", ctypes.c_int64), ("N", ctypes.c_int64), ("K", ctypes.c_int64),
                ("A", ctypes.c_void_p), ("lda", ctypes.c_int64), ("a_mcontig", ctypes.c_bool),
                ("a_f32", ctypes.c_bool), ("B", ctypes.c_void_p), ("ldb", ctypes.c_int64),
                ("b_ncontig", ctypes.c_bool), ("sym", ctypes.c_bool), ("C", ctypes.c_void_p),
                ("ldc", ctypes.c_int64)]


@functools.lru_cache(None)
def symbols():
    out = subprocess.run(["nm", "-D", "--defined-only", _lib.LIB_PATH], capture_output=True,
                         text=True, check=True).stdout
    names = [ln.split()[-1] for ln in out.splitlines() if " T " in ln]
    plain = subprocess.run(["c++filt"], input="\n".join(names), capture_output=True, text=True,
                           check=True).stdout.splitlines()
    return {p.split("(")[0]: n for p, n in zip(plain, names)}


def function(name, restype, *argtypes):
    f = getattr(_lib.lib(), symbols()["mcnla::" + name])
    f.restype, f.argtypes = restype, argtypes
    return f


def args(A, B=None, C=None):
    """A: a device matrix (M x K); B: (K x N) row-major FP64, None: C = A A'."""
    a = ResidueArgs()
    a.M, a.K = A.shape
    a.A, a.lda = A.ptr, A.ld
    a.a_mcontig, a.a_f32 = A.order == "F", A.dtype == np.float32
    a.b_ncontig, a.sym = True, B is None
    a.N = a.M if B is None else B.shape[1]
    if B is not None:
        a.B, a.ldb = B.ptr, B.ld
    if C is not None:
        a.C = C.ptr
    a.ldc = a.N
    return a


def workspace(a, limit):
    """Bytes of the plan taken within `limit` (0: none)."""
    return function("residue_bytes", ctypes.c_size_t, ctypes.POINTER(ResidueArgs), ctypes.c_size_t,
                    ctypes.c_void_p)(ctypes.byref(a), limit, None)


def product(A, B=None, limit=2 << 30):
    """(C, flag) by residues in a workspace of at most `limit` bytes."""
    m, n = A.shape[0], A.shape[0] if B is None else B.shape[1]
    C = mc.DeviceArray.from_numpy(np.full((m, n), np.nan), order="C")
    a = args(A, B, C)
    size = workspace(a, limit)
    assert 0 < size <= limit
    ws = mc.DeviceArray((size // 8 + 32,))
    flag = mc.DeviceArray.from_numpy(np.full(2, np.nan))
    function("gemm_residue", None, ctypes.POINTER(ResidueArgs), ctypes.c_void_p, ctypes.c_size_t,
             ctypes.c_void_p, ctypes.c_void_p)(ctypes.byref(a), ws.ptr, size, flag.ptr, None)
    mc.synchronize()
    return C.numpy(), int(flag.numpy().view(np.int32)[0])


def solver_paths(solver):
    """(sketch, Gram): whether the last solve's products ran by residues."""
    s, g = ctypes.c_bool(), ctypes.c_bool()
    function("solver_products_by_residues", None, ctypes.c_void_p, ctypes.c_void_p,
             ctypes.c_void_p)(solver._h, ctypes.byref(s), ctypes.byref(g))
    return s.value, g.value


def sketcher_path(stage):
    """Whether the last run of this sketcher was by residues."""
    return function("sketcher_by_residues", ctypes.c_bool, ctypes.c_void_p)(stage._h)
