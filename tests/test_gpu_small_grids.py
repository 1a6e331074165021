"""Problems of at most one workgroup for every other compute unit: the planner
takes the kernel with half the default's lines per workgroup.  Its outputs are
those of the default geometry bit for bit (the arithmetic of a line does not
depend on how many share its workgroup) and within the suite's bars of the
oracle, for one line, whole and ragged tiles of either geometry, and around the
grid where the rule ends."""
import numpy as np
import pytest

import fftw3_amd as fa
import oracle
from gpu_util import TOL, cdt, inputs_c, inputs_r, rdt

pytestmark = pytest.mark.gpu


def entry(prec, L, mode, io):
    e = [e for e in fa.catalog() if (e["prec"], e["L"], e["mode"], e["io"], e["variant"]) ==
         (prec, L, mode, io, 0)]
    assert len(e) == 1
    return e[0]


def both(e, plan, run):
    """outputs with the planner's choice and with entry e forced"""
    out = []
    for i in (-1, e["index"]):
        fa.force_kernel(i)
        try:
            p = plan()
        finally:
            fa.force_kernel(-1)
        out.append(run(p))
        p.destroy()
    return out


@pytest.mark.parametrize("prec", ["double", "float"])
@pytest.mark.parametrize("n", [240, 256, 1024, 2048])
@pytest.mark.parametrize("mode", ["row", "col", "r2c", "c2r"])
def test_half_the_lines(eng, prec, n, mode):
    real = mode in ("r2c", "c2r")
    e = entry(prec, n // 2 if real else n, "col" if mode == "col" else "row",
              mode if real else "plain")
    nl, m = e["nl"], n // 2 + 1
    for h in sorted({1, max(1, nl // 2), nl - 1 or 1, nl + 1, 2 * nl + 1, 127 * nl + 1, 128 * nl,
                     128 * nl + 1}):
        if n * h > 1 << 21:
            continue
        if mode == "r2c":
            x = inputs_r(n * h, h, prec)
            ref = oracle.rfftn(x.astype(np.float64).reshape(h, n), axes_batch=1).reshape(-1)
            size, dt = h * m, cdt(prec)
        elif mode == "c2r":
            x = oracle.rfftn(inputs_r(n * h, h, prec).astype(np.float64).reshape(h, n),
                             axes_batch=1).reshape(-1).astype(cdt(prec))
            ref = np.fft.irfft(x.astype(np.complex128).reshape(h, m), n).reshape(-1) * n
            size, dt = h * n, rdt(prec)
        else:
            x = inputs_c(n * h, h, prec)
            z = x.astype(np.complex128)
            ref = (oracle.fftn(z.reshape(n, h).T.copy(), -1, axes_batch=1).T if mode == "col" else
                   oracle.fftn(z.reshape(h, n), -1, axes_batch=1)).reshape(-1)
            size, dt = h * n, cdt(prec)
        a = fa.DeviceBuffer.from_array(x)
        b = fa.DeviceBuffer.from_array(np.zeros(size, dt))

        def plan():
            if mode == "r2c":
                return fa.plan_many_dft_r2c(prec, [n], h, a.ptr, None, 1, n, b.ptr, None, 1, m)
            if mode == "c2r":
                return fa.plan_many_dft_c2r(prec, [n], h, a.ptr, None, 1, m, b.ptr, None, 1, n)
            s, d = (h, 1) if mode == "col" else (1, n)
            return fa.plan_many_dft(prec, [n], h, a.ptr, None, s, d, b.ptr, None, s, d, -1)

        def run(p):
            a.upload(x)
            p.execute()
            return b.download(dt, size)

        y, yd = both(e, plan, run)
        assert np.array_equal(y, yd), (h, nl)
        assert oracle.rel_l2(y, ref) <= TOL[prec], (h, nl)
