"""The SVD of one dense block by the library's own C++ entry (su2::jacobi_svd_batched), below the
truncation, which drops zero blocks and reports neither sweeps nor convergence.  An error would
end the process (a C++ exception has no Python frame to land in): only for blocks that converge.
"""
import ctypes as C

import numpy as np

from su2dmrg_amd import lib as L

_so = C.CDLL(L.lib._name)   # its dependencies' symbols resolve through it, the HIP runtime's too
_fn = _so["_ZN3su218jacobi_svd_batchedERNS_7ContextERSt6vectorINS_11JacobiBlockESaIS3_EEdiiiPdib"]
_fn.restype = C.c_int
_fn.argtypes = [C.c_void_p, C.c_void_p, C.c_double, C.c_int, C.c_int, C.c_int,
                C.POINTER(C.c_double), C.c_int, C.c_bool]


class _Vector(C.Structure):   # std::vector: begin, end, end of storage
    _fields_ = [("begin", C.c_void_p), ("end", C.c_void_p), ("cap", C.c_void_p)]


class _Block(C.Structure):    # su2::JacobiBlock
    _fields_ = [("A", C.c_void_p), ("m", C.c_int), ("n", C.c_int), ("W", C.c_void_p),
                ("V", C.c_void_p), ("s", _Vector), ("group", C.c_int)]


def _hip(name, *args):
    assert _so[name](*args) == 0, name


class _Dev:
    """Device memory of n doubles."""

    def __init__(self, n):
        self.n, p = n, C.c_void_p()
        _hip("hipMalloc", C.byref(p), C.c_size_t(8 * n))
        self.p = p.value

    def put(self, a):
        a = np.asarray(a, dtype=np.float64).ravel(order="F")
        _hip("hipMemcpy", C.c_void_p(self.p), a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes), 1)
        return self

    def get(self, rows):
        a = np.empty(self.n)
        _hip("hipMemcpy", a.ctypes.data_as(C.c_void_p), C.c_void_p(self.p), C.c_size_t(a.nbytes), 2)
        return a.reshape((rows, -1), order="F")

    def __del__(self):
        _so["hipFree"](C.c_void_p(self.p))


def decompose(ctx, mats, plain=False, precondition=256, block=32, inner=1):
    """[(W, V, s)] of the matrices, the sweep count and the largest overlap left (0: converged).
    W = A V for m >= n, A^T V else; columns by ascending singular value s."""
    blocks = (_Block * len(mats))()
    bufs = []
    for b, a in zip(blocks, mats):
        m, n = a.shape
        big, k = max(m, n), min(m, n)
        dev = (_Dev(m * n).put(a), _Dev(big * k), _Dev(k * k))
        bufs.append(dev)
        b.A, b.W, b.V = (x.p for x in dev)
        b.m, b.n = m, n
    vec = _Vector(C.addressof(blocks), C.addressof(blocks) + C.sizeof(blocks),
                  C.addressof(blocks) + C.sizeof(blocks))
    worst = C.c_double(-1.0)
    sweeps = _fn(ctx.h, C.addressof(vec), 1e-13, 60, block, inner, C.byref(worst), precondition,
                 plain)
    ctx.sync()
    out = []
    for b, (_, w, v) in zip(blocks, bufs):
        k = min(b.m, b.n)
        assert b.s.end - b.s.begin == 8 * k
        s = np.array((C.c_double * k).from_address(b.s.begin))
        out.append((w.get(max(b.m, b.n)), v.get(k), s))
    return out, sweeps, worst.value
