"""Whole lines strided on one side only, of lengths without a transposed-store
kernel: two passes on large arrays, one on small ones, against numpy at the
suite's bars; and the allocation-free execute of a plan whose two passes would
need more scratch than it has."""
import ctypes

import numpy as np
import pytest

import fftw3_amd as fa
import oracle
from gpu_util import TOL, cdt, inputs_c

pytestmark = pytest.mark.gpu


# (prec, n, MiB, passes with strided stores, with strided loads): lines a workgroup
# FP32 900 two, 1728 one, 648 three, 1008 four, 784 five; FP64 1728 one, 648 three;
# 225 has no split that ends in a transposed store
@pytest.mark.parametrize("prec,n,mib,st,ld", [
    ("float", 900, 4, 1, 1), ("float", 900, 8, 1, 2), ("float", 900, 66, 2, 2),
    ("float", 1728, 4, 1, 1), ("float", 1728, 17, 2, 2), ("float", 648, 16, 1, 2),
    ("float", 648, 24, 2, 2), ("float", 784, 32, 2, 1), ("float", 225, 66, 1, 1),
    ("float", 1008, 130, 2, 1), ("double", 1728, 4, 1, 1), ("double", 1728, 16, 1, 2),
    ("double", 1728, 66, 2, 2), ("double", 648, 32, 2, 1)])
@pytest.mark.parametrize("side", ["store", "load"])
@pytest.mark.parametrize("sign", [-1, 1])
def test_transposing(eng, prec, n, mib, st, ld, side, sign):
    size = np.dtype(cdt(prec)).itemsize
    h = (mib << 20) // (n * size)
    passes = st if side == "store" else ld
    x = inputs_c(n * h, n, prec)
    a = fa.DeviceBuffer.from_array(x)
    b = fa.DeviceBuffer(x.nbytes)
    u, t = (1, n), (h, 1)
    i, o = (u, t) if side == "store" else (t, u)
    p = fa.plan_many_dft(prec, [n], h, a.ptr, None, i[0], i[1], b.ptr, None, o[0], o[1], sign)
    assert p.npasses() == passes
    lines = x.reshape(h, n) if side == "store" else x.reshape(n, h).T
    z = lines.astype(np.complex128)
    ref = np.fft.fft(z, axis=1) if sign < 0 else np.fft.ifft(z, axis=1) * n
    ref = ref.T if side == "store" else ref
    p.execute()
    got = b.download(cdt(prec), n * h).reshape(ref.shape)
    assert oracle.rel_l2(got.reshape(-1), np.ascontiguousarray(ref).reshape(-1)) <= TOL[prec]
    if mib > 128:
        L = fa.lib()
        L.fftw_amd_execute_noalloc.argtypes = [ctypes.c_void_p] * 3
        b.upload(np.zeros(n * h, cdt(prec)))
        assert L.fftw_amd_execute_noalloc(p.h, a.ptr, b.ptr) == 0
        got = b.download(cdt(prec), n * h).reshape(ref.shape)
        assert oracle.rel_l2(got.reshape(-1), np.ascontiguousarray(ref).reshape(-1)) <= TOL[prec]
    p.destroy()
