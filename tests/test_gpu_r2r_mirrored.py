"""The fused real-to-real kernels' ways to their data: four or two neighbouring
reals at a time (unit stride, aligned arrays, lines a whole number of quads or
pairs apart), one real at a time (any of that missing, at planning or only in
the arrays given at execute), lengths whose radices allow no mirrored stages,
and the non-temporal loads of large inputs.  Every line against the oracle,
relative L2 within the suite's bars (1e-13 FP64, 2e-6 FP32)."""
import numpy as np
import pytest

import fftw3_amd as fa
import oracle
from gpu_util import TOL, rdt

pytestmark = pytest.mark.gpu

KINDS = {"e10": fa.FFTW_REDFT10, "o10": fa.FFTW_RODFT10, "e01": fa.FFTW_REDFT01,
         "o01": fa.FFTW_RODFT01, "e11": fa.FFTW_REDFT11, "o11": fa.FFTW_RODFT11,
         "r2hc": fa.FFTW_R2HC, "hc2r": fa.FFTW_HC2R, "e00": fa.FFTW_REDFT00,
         "o00": fa.FFTW_RODFT00}


# n = 2L: 32 (two threads a line), 96 (three), 90 (odd L, no mirrored stages),
# 26 (odd first radix), 640 and 4096 (whole and several waves a line)
@pytest.mark.parametrize("prec", ["double", "float"])
@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("pad,shift", [(0, 0), (1, 0), (2, 0), (4, 0), (0, 1), (0, 2)])
def test_alignments(eng, prec, kind, pad, shift):
    """Lines n + pad reals apart, arrays shift reals past an aligned start."""
    rs = np.dtype(rdt(prec)).itemsize
    for n in (26, 32, 90, 96, 640, 4096):
        if kind == "e00":
            n += 1
        elif kind == "o00":
            n -= 1
        h, d = 5, n + pad
        x = oracle.uniform(d * h + shift, 900 + n + pad).astype(rdt(prec))
        a = fa.DeviceBuffer.from_array(x)
        b = fa.DeviceBuffer.from_array(np.zeros_like(x))
        p = fa.plan_many_r2r(prec, [n], h, a.ptr + shift * rs, None, 1, d, b.ptr + shift * rs,
                             None, 1, d, [KINDS[kind]])
        p.execute()
        y = b.download(rdt(prec))
        lines = np.stack([x[shift + i * d: shift + i * d + n] for i in range(h)]).astype(np.float64)
        got = np.stack([y[shift + i * d: shift + i * d + n] for i in range(h)])
        ref = np.asarray(oracle.r2rn(lines, [KINDS[kind]], axes_batch=1)).reshape(h, n)
        for i in range(h):
            err = oracle.rel_l2(got[i], ref[i])
            assert err <= TOL[prec], (n, i, err)
        gaps = np.concatenate([y[:shift]] + [y[shift + i * d + n: shift + (i + 1) * d]
                                             for i in range(h)])
        assert not np.any(gaps)
        p.destroy()


@pytest.mark.parametrize("prec", ["double", "float"])
@pytest.mark.parametrize("kind", ["e01", "o01", "e11", "o11", "e00", "o00"])
def test_less_aligned_arrays_at_execute(eng, prec, kind):
    """Planned on aligned arrays, executed on arrays one real further: these
    kinds ask for no more than one real's alignment."""
    n, h = 512, 7
    rs = np.dtype(rdt(prec)).itemsize
    x = oracle.uniform(n * h + 1, 31).astype(rdt(prec))
    a = fa.DeviceBuffer.from_array(x)
    b = fa.DeviceBuffer.from_array(np.zeros_like(x))
    p = fa.plan_many_r2r(prec, [n], h, a.ptr, None, 1, n, b.ptr, None, 1, n, [KINDS[kind]])
    for s in (0, 1):
        p.execute_r2r(a.ptr + s * rs, b.ptr + s * rs)
        y = b.download(rdt(prec))[s:s + n * h].reshape(h, n)
        ref = oracle.r2rn(x[s:s + n * h].astype(np.float64).reshape(h, n), [KINDS[kind]], axes_batch=1)
        assert oracle.rel_l2(y, np.asarray(ref).reshape(h, n)) <= TOL[prec]
    p.destroy()


@pytest.mark.parametrize("prec,n,h", [("float", 2048, 4), ("double", 2048, 2)])
def test_large_first_pass(eng, prec, n, h):
    """A 2-D REDFT10 whose input is 64 MiB: the row pass streams it."""
    x = oracle.uniform(n * n * h, 5).astype(rdt(prec))
    a = fa.DeviceBuffer.from_array(x)
    b = fa.DeviceBuffer(x.nbytes)
    k = [fa.FFTW_REDFT10, fa.FFTW_REDFT10]
    p = fa.plan_many_r2r(prec, [n, n], h, a.ptr, None, 1, n * n, b.ptr, None, 1, n * n, k)
    p.execute()
    y = b.download(rdt(prec)).reshape(h, n, n)
    for i in (0, h - 1):
        ref = oracle.r2rn(x.reshape(h, n, n)[i:i + 1].astype(np.float64), k, axes_batch=1)
        assert oracle.rel_l2(y[i], np.asarray(ref).reshape(n, n)) <= TOL[prec]
    p.destroy()
