"""In-place r2c and c2r whose real and complex lines do not share rows: packed
rows (the complex ones drift over the next real ones) and lines with the batch
innermost.  Every output line lies on other lines' inputs, so the transform has
to read all of them before it writes.  Half-length kernels (540 = 2 * 270,
512 = 2 * 256), a full-length odd one (27) and a length without either (2 * 1155),
against the oracle at the suite's bars; the padded rows that in-place transforms
normally use keep their one-pass kernel."""
import numpy as np
import pytest

import fftw3_amd as fa
import oracle
from gpu_util import TOL, cdt, inputs_r, rdt

pytestmark = pytest.mark.gpu


def layout(n, h, how):
    """(real stride, real dist), (complex stride, complex dist)"""
    m = n // 2 + 1
    return ((1, n), (1, m)) if how == "packed" else ((h, 1), (h, 1))


def positions(n, h, s, d):
    return (np.arange(h)[:, None] * d + np.arange(n)[None, :] * s).reshape(-1)


@pytest.mark.parametrize("prec", ["double", "float"])
@pytest.mark.parametrize("how", ["packed", "inner"])
@pytest.mark.parametrize("n", [27, 512, 540, 2310])
@pytest.mark.parametrize("h", [5, 300])
def test_lines_on_other_lines(eng, prec, how, n, h):
    m = n // 2 + 1
    (rs, rd), (cs, cd) = layout(n, h, how)
    x = inputs_r(h * n, n + h, prec)
    X = oracle.rfftn(x.astype(np.float64).reshape(h, n), axes_batch=1).reshape(h, m)
    pr, pc = positions(n, h, rs, rd), positions(m, h, cs, cd)
    size = max(pr.max() + 1, 2 * (pc.max() + 1))
    size += size % 2
    # forward
    a = np.zeros(size, rdt(prec))
    a[pr] = x
    b = fa.DeviceBuffer.from_array(a)
    p = fa.plan_many_dft_r2c(prec, [n], h, b.ptr, None, rs, rd, b.ptr, None, cs, cd)
    p.execute()
    y = b.download(cdt(prec), size // 2)[pc]
    assert oracle.rel_l2(y, X.reshape(-1)) <= TOL[prec]
    p.destroy()
    # backward
    c = np.zeros(size // 2, cdt(prec))
    c[pc] = X.reshape(-1).astype(cdt(prec))
    ref = oracle.irfftn(c[pc].astype(np.complex128).reshape(h, m), n, axes_batch=1).reshape(-1)
    b.upload(c)
    p = fa.plan_many_dft_c2r(prec, [n], h, b.ptr, None, cs, cd, b.ptr, None, rs, rd)
    p.execute()
    y = b.download(rdt(prec), size)[pr]
    assert oracle.rel_l2(y, ref) <= TOL[prec]
    p.destroy()


@pytest.mark.parametrize("prec", ["double", "float"])
def test_padded_rows_stay_one_pass(eng, prec):
    n, h = 540, 40
    m = n // 2 + 1
    b = fa.DeviceBuffer(2 * m * h * 16)
    for p in (fa.plan_many_dft_r2c(prec, [n], h, b.ptr, None, 1, 2 * m, b.ptr, None, 1, m),
              fa.plan_many_dft_c2r(prec, [n], h, b.ptr, None, 1, m, b.ptr, None, 1, 2 * m),
              fa.plan_many_dft_r2c(prec, [n], 1, b.ptr, None, 3, 1, b.ptr, None, 2, 1)):
        assert p.npasses() == 1
        p.destroy()
