"""The index arithmetic that kernels and tests share (fk_args.h): quotients by
multiplication below 2^31 and through FP64 above, and a line number's batch
indices through either, against integer division: at multiples of the divisor and
their neighbours, powers of two and theirs, and the ends of the ranges."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fftw3_amd", "csrc")
SRC = r"""
#include <stdio.h>
#include <string.h>
#include "fk_args.h"
static unsigned long long seed = 1;
static unsigned long long rnd(void) { return (seed = seed * 6364136223846793005ull + 1442695040888963407ull) >> 11; }
static long long bad, seen;
static void quot(long long q, long long d)
{
    unsigned m, s;
    if (q < 0 || q >> 53) return;
    ++seen;
    if (fk_div_large(q, d) != q / d) ++bad;
    if (q >> 31 || d >> 31) return;
    fk_magic((unsigned long long)d, &m, &s);
    if (fk_div_small((unsigned)q, m, s) != q / d) ++bad;
}
static void lines(long long n0, long long n1, long long n2)
{
    const long long n = n0 * n1 * n2;
    fk_args a;
    int small, i;
    memset(&a, 0, sizeof(a));
    a.nb[0] = n0;
    a.nb[1] = n1;
    a.nb[2] = n2;
    for (small = 0; small < 2; ++small) {
        if (small) {
            if (n >> 31) return;
            fk_magic((unsigned long long)n0, &a.qm[0], &a.qs[0]);
            fk_magic((unsigned long long)n1, &a.qm[1], &a.qs[1]);
        }
        for (i = 0; i < 60; ++i) {
            const long long c[6] = {0, n - 1, n0 * (long long)(rnd() % (n1 * n2)),
                                    n0 * n1 * (long long)(rnd() % n2), (long long)(rnd() % n),
                                    (1ll << (i % 53)) - 1};
            int j, e;
            for (j = 0; j < 6; ++j)
                for (e = -1; e <= 1; ++e) {
                    const long long q = c[j] + e;
                    fk_line r;
                    if (q < 0 || q >= n) continue;
                    r = fk_line_ix(&a, q);
                    ++seen;
                    if (r.i0 != q % n0 || r.i1 != q / n0 % n1 || r.i2 != q / n0 / n1) ++bad;
                }
        }
    }
}
int main(void)
{
    int i, j, e;
    for (i = 0; i < 20000; ++i) {
        const long long d = i < 5000 ? i + 1 : 1 + (long long)(rnd() >> (i % 50));
        for (j = 0; j < 20; ++j) {
            const long long top = (j & 1 ? 1ll << 31 : 1ll << 53) - 1;
            const long long q = j < 2 ? top : j < 12 ? d * (long long)(rnd() % (unsigned long long)(top / d + 1)) : 1ll << (j * 4 - 27);
            for (e = -1; e <= 1; ++e) quot(q + e, d);
        }
    }
    for (i = 0; i < 3000; ++i)
        lines(1 + rnd() % (i % 3 ? 5000 : 7), 1 + rnd() % (i % 5 ? 3000 : 2), 1 + rnd() % (i % 2 ? 40 : 4000));
    for (e = -1; e <= 1; ++e) {
        lines((1ll << 31) + e, 1, 1);
        lines(65536, 32768 + e, 1);
        lines(3, 5, (1ll << 40) + e);
        lines((1ll << 33) + e, 7, 11);
    }
    printf("%lld %d\n", bad, seen > 1000000);
    return 0;
}
"""


@pytest.mark.parametrize("opt", ["-O0", "-O2"])
def test_index_arithmetic(tmp_path, opt):
    src = tmp_path / "ix.c"
    src.write_text(SRC)
    exe = str(tmp_path / "ix")
    subprocess.check_call(["gcc", opt, "-I", CSRC, "-o", exe, str(src)])
    assert subprocess.check_output([exe]).split() == [b"0", b"1"]
