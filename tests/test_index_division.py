"""The divisions the kernels index lines and twiddles with, against integer
division: by multiplication (fk_magic, quotients below 2^31) and through FP64
(div_large's two lines, quotients up to 2^53), at the values where a rounding
would show: multiples of the divisor and their neighbours, powers of two and
theirs, the ends of the range."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fftw3_amd", "csrc")
SRC = r"""
#include <stdio.h>
#include "fk_args.h"
static long long div_large(long long q, long long d)
{
    const long long t = (long long)((double)q / (double)d), r = q - t * d;
    return r < 0 ? t - 1 : r >= d ? t + 1 : t;
}
static unsigned long long seed = 1;
static unsigned long long rnd(void) { return (seed = seed * 6364136223846793005ull + 1442695040888963407ull) >> 11; }
static long long bad;
static void magic(unsigned long long q, unsigned long long d, unsigned m, unsigned s)
{
    if (q >> 31) return;
    if ((unsigned)((2ull * q * m) >> 32) >> s != q / d) ++bad;
}
static void large(long long q, long long d)
{
    if (q < 0 || q >> 53) return;
    if (div_large(q, d) != q / d) ++bad;
}
int main(void)
{
    long i, j, e;
    for (i = 0; i < 40000; ++i) {
        const unsigned long long d = i < 20000 ? i + 1 : i < 39000 ? 1 + rnd() % 0x7fffffff : 0x7fffffff - (i - 39000);
        unsigned m, s;
        fk_magic(d, &m, &s);
        for (j = 0; j < 20; ++j) {
            const unsigned long long q = j == 0 ? 0 : j == 1 ? 0x7fffffff : j < 11 ? d * (rnd() % (0x7fffffff / d + 1)) : rnd() >> 22;
            for (e = -1; e <= 1; ++e) magic(q + e, d, m, s);
        }
        for (j = 0; j < 31; ++j)
            for (e = -1; e <= 1; ++e) magic((1ull << j) + e, d, m, s);
        for (j = 0; j < 20; ++j) {
            const long long D = j & 1 ? (long long)d : (long long)(1 + (rnd() >> (j + 1)));
            const long long q = j == 0 ? (1ll << 53) - 1 : D * (long long)(rnd() % (unsigned long long)((1ll << 53) / D));
            for (e = -1; e <= 1; ++e) large(q + e, D);
        }
    }
    printf("%lld\n", bad);
    return 0;
}
"""


@pytest.mark.parametrize("opt", ["-O0", "-O2"])
def test_index_division(tmp_path, opt):
    src = tmp_path / "div.c"
    src.write_text(SRC)
    exe = str(tmp_path / "div")
    subprocess.check_call(["gcc", opt, "-I", CSRC, "-o", exe, str(src)])
    assert subprocess.check_output([exe]).split() == [b"0"]
