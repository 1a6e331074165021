"""Products of 2, 3, 5 and 7 as lines: one pass where the catalog holds the
length (rows, columns, half of an even real line), and longer lines, which are
split into the lengths kept for that.  Relative L2
within the suite's bars (1e-13 FP64, 2e-6 FP32)."""
import re

import numpy as np
import pytest

import fftw3_amd as fa
import oracle
from gpu_util import TOL, c2c_many, cdt, inputs_c, inputs_r

pytestmark = pytest.mark.gpu


def lengths(p):
    return [int(m.group(1)) for i in p.pass_info() for m in [re.search(r" L=(\d+) ", i)] if m]


# the ends of each range: all up to 512, factors 4 or 10 to 1024, 16 or 40 to 2048
@pytest.mark.parametrize("prec", ["double", "float"])
@pytest.mark.parametrize("n", [70, 105, 441, 486, 504, 490, 540, 980, 1008, 1080, 1120, 2000, 2016])
def test_one_pass(eng, prec, n):
    h = 11
    x = inputs_c(n * h, n, prec)
    a = fa.DeviceBuffer.from_array(x)
    b = fa.DeviceBuffer(x.nbytes)
    z = x.astype(np.complex128)
    for s, d in ((1, n), (h, 1)):
        p = fa.plan_many_dft(prec, [n], h, a.ptr, None, s, d, b.ptr, None, s, d, -1)
        assert lengths(p) == [n]
        p.execute()
        y = b.download(cdt(prec))
        ref = (oracle.fftn(z.reshape(h, n), -1, axes_batch=1) if s == 1 else
               oracle.fftn(z.reshape(n, h).T.copy(), -1, axes_batch=1).T)
        assert oracle.rel_l2(y, np.ascontiguousarray(ref).reshape(-1)) <= TOL[prec], s
        p.destroy()
    m = n + 1
    r = inputs_r(2 * n * h, n + 1, prec)
    a = fa.DeviceBuffer.from_array(r)
    b = fa.DeviceBuffer(h * m * np.dtype(cdt(prec)).itemsize)
    p = fa.plan_many_dft_r2c(prec, [2 * n], h, a.ptr, None, 1, 2 * n, b.ptr, None, 1, m)
    assert lengths(p) == [n]
    p.execute()
    ref = oracle.rfftn(r.astype(np.float64).reshape(h, 2 * n), axes_batch=1).reshape(-1)
    assert oracle.rel_l2(b.download(cdt(prec)), ref) <= TOL[prec]
    p.destroy()


@pytest.mark.parametrize("prec", ["double", "float"])
@pytest.mark.parametrize("n", [3675, 7350, 2268 * 4, 96 * 1920, 444528])
def test_split_lines(eng, prec, n):
    a = fa.DeviceBuffer(16 * n * 2)
    p = fa.plan_many_dft(prec, [n], 2, a.ptr, None, 1, n, a.ptr, None, 1, n, -1)
    for L in lengths(p):
        odd = L
        while odd % 2 == 0:
            odd //= 2
        powers = any(odd == q ** k for q in (3, 5, 7) for k in range(1, 9)) and odd == L
        assert L <= 64 or odd in (1, 3, 5) or powers or L in (100, 1000, 1001, 10000)
    p.destroy()
    y, ref, _ = c2c_many(prec, [n], 2, -1, seed=n % 97)
    assert oracle.rel_l2(y, ref) <= TOL[prec]
