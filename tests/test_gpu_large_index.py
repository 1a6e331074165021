"""The 64-bit branches of the kernels' index arithmetic on the device: a pass of
more than 2^31 lines, and a four-step split of 2^31 points, every output
checked on the device.  The checks use torch, which has to be loaded before the
engine's library: each case is a process of its own."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
pytestmark = pytest.mark.gpu

HEAD = r"""
import sys
sys.path.insert(0, %r)
import torch
import fftw3_amd as fa
def room(gib):
    if torch.cuda.mem_get_info()[0] < gib << 30:
        print("no room", flush=True)
        sys.exit(0)
""" % ROOT

LINES = HEAD + r"""
# 2-point FP32 lines in place: outputs are x0 + x1 and x0 - x1, exactly (inputs are
# small whole numbers)
room(48)
lines, chunk = (1 << 31) + 77, 1 << 26
x = torch.empty(lines, 2, dtype=torch.complex64, device="cuda")
def inputs(lo, hi):
    i = torch.arange(lo, hi, device="cuda")
    r = torch.stack([i % 1021, i % 4093, (i >> 7) % 2039, (i >> 20) % 8191], 1).float()
    return torch.view_as_complex(r.reshape(-1, 2, 2).contiguous())
for lo in range(0, lines, chunk):
    x[lo:lo + chunk] = inputs(lo, min(lines, lo + chunk))
torch.cuda.synchronize()
fa.init()
p = fa.plan_guru_dft("float", [(2, 1, 1)], [(lines, 2, 2)], x.data_ptr(), x.data_ptr(), -1, wide=True)
assert p.npasses() == 1 and "lines=%d" % lines in p.pass_info()[0], p.pass_info()
print("planned", p.pass_info(), flush=True)
p.execute()
for lo in range(0, lines, chunk):
    z, y = inputs(lo, min(lines, lo + chunk)), x[lo:lo + chunk]
    assert torch.equal(y[:, 0], z[:, 0] + z[:, 1]) and torch.equal(y[:, 1], z[:, 0] - z[:, 1]), lo
print("checked", flush=True)
"""

SPLIT = HEAD + r"""
# one FP32 transform of 2^31 points of an input with three nonzero samples, against
# its closed form in FP64 (k * i mod n is exact in 64 bits)
room(80)
n, chunk = 1 << 31, 1 << 26
at, amp = [1, 123456789, n - 3], [1.0, -0.5, 0.75]
x = torch.zeros(n, dtype=torch.complex64, device="cuda")
for i, v in zip(at, amp):
    x[i] = v
torch.cuda.synchronize()
fa.init()
p = fa.plan_guru_dft("float", [(n, 1, 1)], [], x.data_ptr(), x.data_ptr(), -1, wide=True)
assert p.npasses() >= 2
print("planned", p.pass_info(), flush=True)
p.execute()
err = 0.0
for lo in range(0, n, chunk):
    k = torch.arange(lo, lo + chunk, device="cuda")
    ref = torch.zeros(chunk, dtype=torch.complex128, device="cuda")
    for i, v in zip(at, amp):
        ang = ((k * i) & (n - 1)).double() * (-2 * torch.pi / n)
        ref += v * torch.polar(torch.ones_like(ang), ang)
    err = max(err, float((x[lo:lo + chunk].to(torch.complex128) - ref).abs().max()))
# three terms of 2.25 together, each through at most 4 rounded twiddle products and
# 31 additions in FP32
assert err <= 35 * 2.0 ** -24 * 2.25, err
print("checked", flush=True)
"""


@pytest.mark.parametrize("script", [LINES, SPLIT], ids=["lines", "split"])
def test_beyond_31_bits(script):
    r = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
    if "no room" in r.stdout:
        pytest.skip("not enough device memory")
    assert "checked" in r.stdout
