"""The work whose speed is tracked, through the public entry points of the
Python binding (the plan / execute C ABI underneath).

Every case is a plan made once with FFTW_ESTIMATE (the binding's default
flag) and executed on new arrays, in asynchronous mode on the default stream,
as a streaming program does.  Kinds:

  c2c    one complex transform (sign -1 or +1), or with sign 0 the forward
         transform x -> y followed by the backward one y -> z (place "out")
         or y -> y (place "in");
  r2c    real to half-complex;
  real   r2c, then c2r of the result back to a real array (multi-dimensional
         c2r destroys its input, so only the real result is an output);
  r2r    a real-to-real transform of the given kind along every dimension,
         and with "inverse" the matching inverse kind of its result;
  batch  1-D complex transforms of several lengths in one batch object.
"""
import math

import numpy as np
import torch

import fftw3_amd as fa

_KIND = {"r2hc": fa.FFTW_R2HC, "hc2r": fa.FFTW_HC2R, "dht": fa.FFTW_DHT,
         "e00": fa.FFTW_REDFT00, "e01": fa.FFTW_REDFT01, "e10": fa.FFTW_REDFT10,
         "e11": fa.FFTW_REDFT11, "o00": fa.FFTW_RODFT00, "o01": fa.FFTW_RODFT01,
         "o10": fa.FFTW_RODFT10, "o11": fa.FFTW_RODFT11}
_INV = {"r2hc": "hc2r", "hc2r": "r2hc", "dht": "dht", "e00": "e00", "e01": "e10", "e10": "e01",
        "e11": "e11", "o00": "o00", "o01": "o10", "o10": "o01", "o11": "o11"}


def _case(kind, prec, shape, howmany, **more):
    c = {"kind": kind, "prec": prec, "shape": "x".join(str(n) for n in shape), "howmany": howmany}
    c.update(more)
    return c


def listed():
    def c(name, *a, **k):
        return dict(_case(*a, **k), name=name)

    return [
        # one short line there and back: what calls cost when the work is nothing
        c("c2c_f32_256", "c2c", "float", [256], 1, sign=0, place="out"),
        # one small volume: three dependent launches that leave most of the chip idle
        c("c2c_f64_64x64x64", "c2c", "double", [64, 64, 64], 1, sign=-1, place="out"),
        # the single-size batch of the benchmark
        c("c2c_f64_4096_b1024", "c2c", "double", [4096], 1024, sign=-1, place="out"),
        # a batch of lines whose length is no power of two, backward
        c("c2c_f32_1920_b8192", "c2c", "float", [1920], 8192, sign=1, place="out"),
        # the long 1-D lines of the precision study
        c("c2c_f32_16777216_b8", "c2c", "float", [1 << 24], 8, sign=-1, place="out"),
        # the benchmark's volume, there and back: the largest call
        c("c2c_f64_512x512x512", "c2c", "double", [512, 512, 512], 1, sign=0, place="out"),
        # the benchmark's real images, forward
        c("r2c_f32_2048x2048_b64", "r2c", "float", [2048, 2048], 64),
        # ... and there and back, as a filter does
        c("real_f32_2048x2048_b64", "real", "float", [2048, 2048], 64),
        # video frames: neither side a power of two
        c("real_f32_1080x1920_b16", "real", "float", [1080, 1920], 16),
        # a field of a double precision solver, there and back
        c("real_f64_256x256x256", "real", "double", [256, 256, 256], 1),
        # the cosine transform of the benchmark's images and its inverse
        c("dct_f32_2048x2048_b16", "r2r", "float", [2048, 2048], 16, r2r="e10", inverse=True),
        # uneven lengths in one batch (powers of two, composites, a prime): the
        # benchmark's set at a quarter of its points
        c("batch_f32_uneven", "batch", "float", [1000, 1001, 2187, 4093, 4096, 65536, 1 << 20], 0,
          counts="13x8x3x182x1x2x63", sign=-1),
    ]


def _length(rng, lo, hi):
    """A transform length in [lo, hi]: a power of two, a product of small
    primes, or any number."""
    t = rng.random()
    x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    if t < 0.4:
        n = 1 << max(0, round(math.log2(x)))
    elif t < 0.85:
        n = 1
        while True:
            p = rng.choice((2, 2, 2, 3, 3, 5, 7))
            if n * p > x:
                break
            n *= p
    else:
        n = int(x)
    return max(lo, min(hi, n))


def draw(rng):
    prec = rng.choice(("float", "float", "double"))
    kind = rng.choice(("c2c", "c2c", "c2c", "c2c", "r2c", "real", "real", "r2r", "r2r", "batch"))
    if kind == "batch":
        k = rng.randint(3, 8)
        shape = [_length(rng, 64, 1 << 20) for _ in range(k)]
        counts = [max(1, min(4096, int((1 << 24) / k / n * rng.random()))) for n in shape]
        return _case("batch", prec, shape, 0, counts="x".join(str(h) for h in counts),
                     sign=rng.choice((-1, 1)))
    points = 1 << 25 if prec == "float" else 1 << 24
    rank = rng.choice((1, 1, 2, 3))
    # the length of one transform, then how many fit the drawn total
    hi = {1: 1 << 22, 2: 4096, 3: 320}[rank]
    if kind == "r2r":
        hi = {1: 1 << 18, 2: 2048, 3: 192}[rank]
    shape = [_length(rng, 8, hi) for _ in range(rank)]
    while math.prod(shape) > points:
        shape[shape.index(max(shape))] //= 2
    n = math.prod(shape)
    h = max(1, int(math.exp(rng.uniform(0.0, math.log(max(1.0, points / n)))) + 0.5))
    if kind == "c2c":
        sign = rng.choice((-1, -1, 1, 0))
        place = rng.choice(("out", "out", "in")) if sign == 0 else "out"
        layout = "columns" if rank == 1 and h > 1 and rng.random() < 0.25 else "lines"
        return _case("c2c", prec, shape, h, sign=sign, place=place, layout=layout)
    if kind == "r2r":
        return _case("r2r", prec, shape, h, r2r=rng.choice(sorted(_KIND)),
                     inverse=rng.random() < 0.5)
    return _case(kind, prec, shape, h)


# ---------------------------------------------------------------------------

def _shape(case):
    return [int(s) for s in case["shape"].split("x")]


def _groups(case):
    return list(zip(_shape(case), [int(s) for s in case["counts"].split("x")]))


def _types(case):
    return (torch.float64, torch.complex128) if case["prec"] == "double" else \
        (torch.float32, torch.complex64)


def _columns(case):
    return case.get("layout") == "columns"


def _inputs(case, seed):
    """Values uniform in [-1, 1), on the GPU, from the seed alone."""
    rt, _ = _types(case)
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def real(*s):
        return torch.rand(s, generator=g, device="cuda", dtype=rt).mul_(2).sub_(1)

    s, h, kind = _shape(case), case["howmany"], case["kind"]
    if kind == "batch":
        return [torch.view_as_complex(real(k, n, 2)) for n, k in _groups(case)]
    if kind == "c2c":
        return torch.view_as_complex(real(s[0], h, 2) if _columns(case) else real(h, *s, 2))
    return real(h, *s)


def prepare(case, seed):
    """Inputs, output arrays and plans that a program keeps."""
    fa.init()
    fa.lib().fftw_amd_set_async(1)
    _, ct = _types(case)
    prec, kind, s, h = case["prec"], case["kind"], _shape(case), case["howmany"]
    x = _inputs(case, seed)
    st = {"kind": kind, "x": x}
    N = math.prod(s)
    if kind == "batch":
        st["y"] = [torch.zeros_like(v) for v in x]
        groups = [(n, k, a.data_ptr(), b.data_ptr())
                  for (n, k), a, b in zip(_groups(case), x, st["y"])]
        torch.cuda.synchronize()
        st["batch"] = fa.Batch(prec, groups, case["sign"])
        st["stream"] = torch.cuda.ExternalStream(st["batch"].stream())
    elif kind == "c2c":
        st["y"] = torch.zeros_like(x)
        stride, dist = (h, 1) if _columns(case) else (1, N)

        def plan(a, b, sign):
            return fa.plan_many_dft(prec, s, h, a.data_ptr(), None, stride, dist,
                                    b.data_ptr(), None, stride, dist, sign)

        if case["sign"]:
            st["plan"] = plan(x, st["y"], case["sign"])
        else:
            st["plan"] = plan(x, st["y"], fa.FFTW_FORWARD)
            st["z"] = torch.zeros_like(x) if case["place"] == "out" else st["y"]
            st["back"] = plan(st["y"], st["z"], fa.FFTW_BACKWARD)
    elif kind in ("r2c", "real"):
        nh = s[-1] // 2 + 1
        st["y"] = torch.zeros([h] + s[:-1] + [nh], dtype=ct, device="cuda")
        M = N // s[-1] * nh
        st["plan"] = fa.plan_many_dft_r2c(prec, s, h, x.data_ptr(), None, 1, N,
                                          st["y"].data_ptr(), None, 1, M)
        if kind == "real":
            st["z"] = torch.zeros_like(x)
            st["back"] = fa.plan_many_dft_c2r(prec, s, h, st["y"].data_ptr(), None, 1, M,
                                              st["z"].data_ptr(), None, 1, N)
    else:
        def plan(a, b, name):
            return fa.plan_many_r2r(prec, s, h, a.data_ptr(), None, 1, N, b.data_ptr(), None, 1, N,
                                    [_KIND[name]] * len(s))

        st["y"] = torch.zeros_like(x)
        st["plan"] = plan(x, st["y"], case["r2r"])
        if case["inverse"]:
            st["z"] = torch.zeros_like(x)
            st["back"] = plan(st["y"], st["z"], _INV[case["r2r"]])
    return st


def run(st):
    kind = st["kind"]
    if kind == "batch":
        # the batch runs on its own stream: ordered after what was queued
        # here, and what follows here after it
        now = torch.cuda.current_stream()
        st["stream"].wait_stream(now)
        st["batch"].execute()
        now.wait_stream(st["stream"])
        return st["y"]
    x, y = st["x"].data_ptr(), st["y"].data_ptr()
    if kind == "c2c":
        st["plan"].execute_dft(x, y)
        if "back" not in st:
            return st["y"]
        st["back"].execute_dft(y, st["z"].data_ptr())
        return [st["y"], st["z"]] if st["z"] is not st["y"] else st["z"]
    if kind == "r2c":
        st["plan"].execute_r2c(x, y)
        return st["y"]
    if kind == "real":
        st["plan"].execute_r2c(x, y)
        st["back"].execute_c2r(y, st["z"].data_ptr())
        return st["z"]
    st["plan"].execute_r2r(x, y)
    if "back" not in st:
        return st["y"]
    st["back"].execute_r2r(y, st["z"].data_ptr())
    return [st["y"], st["z"]]


def work(case):
    s, h, kind = _shape(case), case["howmany"], case["kind"]
    rs = 8 if case["prec"] == "double" else 4
    if kind == "batch":
        g = _groups(case)
        return {"bytes": 4.0 * rs * sum(n * k for n, k in g),
                "flops": 5.0 * sum(n * k * math.log2(max(2, n)) for n, k in g)}
    N = math.prod(s)
    lg = math.log2(max(2, N))
    if kind == "c2c":
        runs = 1 if case["sign"] else 2
        return {"bytes": 4.0 * rs * N * h * runs, "flops": 5.0 * N * h * lg * runs}
    if kind == "r2r":
        runs = 2 if case["inverse"] else 1
        return {"bytes": 2.0 * rs * N * h * runs, "flops": 2.5 * N * h * lg * runs}
    runs = 2 if kind == "real" else 1
    half = N // s[-1] * (s[-1] // 2 + 1)
    return {"bytes": (rs * N + 2.0 * rs * half) * h * runs, "flops": 2.5 * N * h * lg * runs}


# ---------------------------------------------------------------------------
# the same in 64 bits

def _fft(x, dims, sign):
    if sign < 0:
        return torch.fft.fftn(x, dim=dims)
    return torch.fft.ifftn(x, dim=dims, norm="forward")


def _phase(e):
    return torch.polar(torch.ones_like(e), e)


def _r2r_last(x, kind):
    """FFTW's definition of an r2r kind along the last dim, through a
    zero-padded complex FFT (doc/reference.texi:2021-2350)."""
    n = x.shape[-1]
    j = torch.arange(n, dtype=torch.float64)
    if kind == "r2hc":
        f = torch.fft.fft(x, dim=-1)
        return torch.cat([f.real[..., :n // 2 + 1], f.imag[..., 1:(n + 1) // 2].flip(-1)], -1)
    if kind == "dht":
        f = torch.fft.fft(x, dim=-1)
        return f.real - f.imag
    if kind == "hc2r":
        half = torch.zeros(x.shape[:-1] + (n // 2 + 1,), dtype=torch.complex128)
        half.real.copy_(x[..., :n // 2 + 1])
        half.imag[..., 1:(n + 1) // 2] = x[..., n // 2 + 1:].flip(-1)
        return torch.fft.irfft(half, n=n, dim=-1, norm="forward")
    m = {"e00": 2 * (n - 1), "o00": 2 * (n + 1)}.get(kind, 2 * n)
    if kind == "e00":
        z = x.clone()
        z[..., 0] *= 0.5
        z[..., -1] *= 0.5
        return 2 * torch.fft.fft(z, n=m, dim=-1).real[..., :n]
    if kind == "o00":
        z = torch.nn.functional.pad(x, (1, 0))
        return -2 * torch.fft.fft(z, n=m, dim=-1).imag[..., 1:n + 1]
    if kind in ("e10", "o10"):
        o = 0 if kind == "e10" else 1
        f = torch.fft.fft(x, n=m, dim=-1)[..., o:o + n] * _phase(-math.pi * (j + o) / (2 * n))
        return 2 * f.real if kind == "e10" else -2 * f.imag
    if kind == "e01":
        z = x * _phase(-math.pi * j / (2 * n))
        z[..., 0] *= 0.5
        return 2 * torch.fft.fft(z, n=m, dim=-1).real[..., :n]
    if kind == "o01":
        z = x * _phase(-math.pi * (j + 1) / (2 * n))
        z[..., -1] *= 0.5
        z = torch.nn.functional.pad(z, (1, 0))
        return -2 * torch.fft.fft(z, n=m, dim=-1).imag[..., :n]
    f = torch.fft.fft(x * _phase(-math.pi * j / (2 * n)), n=m, dim=-1)[..., :n]
    f = f * _phase(-math.pi * (2 * j + 1) / (4 * n))
    return 2 * f.real if kind == "e11" else -2 * f.imag


def _r2r(x, rank, kind):
    for d in range(x.dim() - rank, x.dim()):
        x = _r2r_last(x.transpose(d, -1), kind).transpose(d, -1)
    return x


def exact(case, seed):
    s, kind = _shape(case), case["kind"]
    x = _inputs(case, seed)
    if kind == "batch":
        return [_fft(v.cpu().to(torch.complex128), (1,), case["sign"]) for v in x]
    dims = (0,) if _columns(case) else tuple(range(1, len(s) + 1))
    if kind == "c2c":
        x = x.cpu().to(torch.complex128)
        if case["sign"]:
            return _fft(x, dims, case["sign"])
        back = x * float(math.prod(s))
        return [_fft(x, dims, -1), back] if case["place"] == "out" else back
    x = x.cpu().to(torch.float64)
    if kind == "r2c":
        return torch.fft.rfftn(x, dim=dims)
    if kind == "real":
        return x * float(math.prod(s))
    y = _r2r(x, len(s), case["r2r"])
    if not case["inverse"]:
        return y
    scale = math.prod({"e00": 2 * (n - 1), "o00": 2 * (n + 1)}.get(
        case["r2r"], n if case["r2r"] in ("r2hc", "hc2r", "dht") else 2 * n) for n in s)
    return [y, x * float(scale)]
