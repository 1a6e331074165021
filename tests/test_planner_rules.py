"""The planner's own rules on the CPU: a C program that includes the engine's
source and runs its planning functions on the built catalog, without a device
(no array, table or launch is made)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "fftw3_amd")
ROCM = "/opt/rocm"

HEAD = r"""
#include "engine.c"
static long long bad, seen;
#define CHECK(c, ...) do { ++seen; if (!(c) && bad++ < 20) printf(__VA_ARGS__); } while (0)
static void start(void) { g_reg = fk_registry(&g_nreg); index_catalog(); }
static fk_plan *begin(ctx *c, int prec)
{
    fk_plan *P = (fk_plan *)calloc(1, sizeof(fk_plan));
    P->prec = prec;
    memset(c, 0, sizeof(*c));
    c->P = P;
    c->bin = FK_BUF_IN;
    c->bout = FK_BUF_OUT;
    return P;
}
"""


def run(tmp_path, body):
    if not os.path.exists(os.path.join(ROCM, "lib", "libamdhip64.so")):
        pytest.skip("no HIP runtime to link against")
    src = tmp_path / "t.c"
    src.write_text(HEAD + body)
    exe = str(tmp_path / "t")
    subprocess.check_call(["gcc", "-std=gnu11", "-O1", "-w", "-D__HIP_PLATFORM_AMD__",
                           "-I" + os.path.join(PKG, "csrc"), "-I" + os.path.join(ROCM, "include"),
                           "-o", exe, str(src), "-L" + PKG, "-lfftw3_amd", "-L" + ROCM + "/lib",
                           "-lamdhip64", "-lpthread", "-lm", "-Wl,-rpath," + PKG,
                           "-Wl,-rpath," + ROCM + "/lib"])
    out = subprocess.run([exe], capture_output=True, text=True, check=True).stdout
    *msgs, last = out.strip().split("\n")
    bad, seen = map(int, last.split())
    assert bad == 0, "\n".join(msgs)
    assert seen > 0
    return seen


def test_stored_choice_is_the_same_kernel_on_any_device(tmp_path):
    """A decision vector made on one device names the same kernels on another:
    for every catalog key with alternatives, the default picked with 256, 64 and
    8 compute units and every explicit choice resolve to the same entry wherever
    they are replayed."""
    run(tmp_path, r"""
int main(void)
{
    static const int ncu[] = {256, 64, 8};
    static const long long lines[] = {0, 1, 3, 16, 100, 700, 5000, 1LL << 33};
    int i, a, b, l;
    start();
    for (i = 0; i < g_nreg; ++i) {
        const fk_kernel *k = g_reg + i, *vs[16];
        int n = find_variants(k->prec, k->L, k->mode, k->io, vs, 16), v;
        if (k->variant || n < 2) continue;
        for (l = 0; l < 8; ++l)
            for (a = 0; a < 3; ++a)
                for (v = -1; v < n; ++v) {
                    const fk_kernel *first;
                    ctx c;
                    fk_plan *P = begin(&c, k->prec);
                    int made = v;
                    g_ncu = ncu[a];
                    c.choice = v < 0 ? 0 : &made;
                    c.nchoice = v >= 0;
                    first = pick_variant(&c, k->prec, k->L, k->mode, k->io, lines[l]);
                    made = P->choice[0];
                    CHECK(v < 0 || first == vs[v], "L=%d choice %d\n", k->L, v);
                    for (b = 0; b < 3; ++b) {
                        ctx d;
                        fk_plan *Q = begin(&d, k->prec);
                        g_ncu = ncu[b];
                        d.choice = &made;
                        d.nchoice = 1;
                        CHECK(pick_variant(&d, k->prec, k->L, k->mode, k->io, lines[l]) == first,
                              "L=%d mode=%d io=%d lines=%lld made at %d CUs, replayed at %d\n", k->L,
                              k->mode, k->io, lines[l], ncu[a], ncu[b]);
                        free(Q);
                    }
                    free(P);
                }
    }
    printf("%lld %lld\n", bad, seen);
    return 0;
}
""")


def test_half_the_lines_where_the_grid_is_small(tmp_path):
    """The default geometry of a pass: half the lines per workgroup exactly where
    the catalog has such a variant, at most every other compute unit would have a
    workgroup, and column runs (transposed stores) stay at 64 bytes; on either
    side of the limit, with whole and ragged last tiles."""
    run(tmp_path, r"""
int main(void)
{
    int i, v, t, half = 0;
    start();
    g_ncu = 256;
    for (i = 0; i < g_nreg; ++i) {
        const fk_kernel *k = g_reg + i, *vs[16], *h = 0;
        int n = find_variants(k->prec, k->L, k->mode, k->io, vs, 16);
        static const long long tiles[] = {1, 2, 127, 128, 129, 256, 4000};
        if (k->variant) continue;
        for (v = 1; v < n && !h; ++v)
            if (!vs[v]->loop && vs[v]->tpl == k->tpl && 2 * vs[v]->nl == k->nl &&
                vs[v]->nrad == k->nrad && !memcmp(vs[v]->rad, k->rad, sizeof(int) * k->nrad))
                h = vs[v];
        for (t = 0; t < 7; ++t) {
            long long end[2] = {tiles[t] * k->nl, tiles[t] * k->nl - k->nl + 1};
            for (v = 0; v < 2; ++v) {
                ctx c;
                fk_plan *P = begin(&c, k->prec);
                const int wide = k->mode == FK_ROW && k->io != FK_IO_TOUT;
                const int run = k->nl * (k->prec ? 8 : 16);
                const int take = h && !k->loop && tiles[t] <= 128 && (wide || run >= 128);
                const fk_kernel *p = pick_variant(&c, k->prec, k->L, k->mode, k->io, end[v]);
                CHECK(p == (take ? h : k), "prec=%d L=%d mode=%d io=%d lines=%lld: nl %d\n",
                      k->prec, k->L, k->mode, k->io, end[v], p->nl);
                half += take;
                free(P);
            }
        }
    }
    CHECK(half > 100, "only %d cases take the half-lines kernel\n", half);
    printf("%lld %lld\n", bad, seen);
    return 0;
}
""")


EMIT = r"""
/* one logical pass of kernel (prec, L, mode, io) over batch dims b, as the
   planner emits it but without its tables */
static void emit(ctx *c, int prec, int L, int io, int nb, const fk_dim *b, int ibuf, int obuf)
{
    fk_pass p;
    memset(&p, 0, sizeof(p));
    p.type = FK_PASS_STOCKHAM;
    p.k = find_kernel(prec, L, FK_ROW, io);
    p.ibuf = ibuf;
    p.obuf = obuf;
    p.a.is = p.a.os = 1;
    emit_loops(c, &p, nb, b, prec ? 8 : 16, prec ? 8 : 16);
}
static unsigned nt(const fk_plan *P, int i) { return P->pass[i].a.flags & (FK_NT_IN | FK_NT_OUT); }
"""


def test_cache_rules_take_a_pass_with_its_loops(tmp_path):
    """Batch dims beyond the three that a launch addresses become several launches
    of one logical pass: all of them get the same cache flags, by the size of the
    whole pass and by whether it is the plan's only or first one."""
    run(tmp_path, EMIT + r"""
int main(void)
{
    int m, one, i;
    start();
    for (one = 0; one < 2; ++one)
        for (m = 1; m <= 1024; m *= 4) {
            /* 512-point FP64 lines, five batch dims that do not merge: 6 * 5
               launches of m * 64 lines */
            fk_dim b[5] = {{8, 520, 520}, {8, 8320, 8320}, {m, 133120, 133120},
                           {6, 133120LL * (m + 1), 133120LL * (m + 1)},
                           {5, 133120LL * (m + 1) * 8, 133120LL * (m + 1) * 8}};
            const long long bytes = 30LL * 64 * m * 512 * 16, MB = 1 << 20;
            unsigned want0;
            int n0;
            ctx c;
            fk_plan *P = begin(&c, 0);
            emit(&c, 0, 512, FK_IO_PLAIN, 5, b, FK_BUF_IN, FK_BUF_OUT);
            n0 = P->npass;
            CHECK(n0 > 1, "one launch only\n");
            if (!one) emit(&c, 0, 512, FK_IO_PLAIN, 5, b, FK_BUF_OUT, FK_BUF_OUT);
            mark_streams(P);
            if (one) want0 = bytes >= 16 * MB ? FK_NT_IN | FK_NT_OUT : 0;
            else want0 = (bytes >= 128 * MB ? FK_NT_IN : 0) | (bytes >= 1024 * MB ? FK_NT_OUT : 0);
            for (i = 0; i < P->npass; ++i)
                CHECK(nt(P, i) == (i < n0 ? want0 : 0), "%s pass, %lld MiB, launch %d of %d: %u\n",
                      one ? "only" : i < n0 ? "first" : "second", bytes / MB, i, P->npass, nt(P, i));
            free(P->pass);
            free(P);
        }
    printf("%lld %lld\n", bad, seen);
    return 0;
}
""")


def test_wide_accesses_need_the_arrays_alignment(tmp_path):
    """Non-temporal accesses of rows whose threads per line are not 16, 32, 64 ...
    only on arrays (with the launch's offset) at 64-byte boundaries, quads at 16 bytes,
    pairs of REDFT11 at two reals; each array decides for its own side, and
    other flags stay."""
    run(tmp_path, EMIT + r"""
int main(void)
{
    static const int ios[] = {FK_IO_PLAIN, FK_IO_PLAIN, FK_IO_PLAIN, FK_IO_R2C_RR, FK_IO_C2R_RR,
                              FK_IO_DCT4};
    static const int Ls[] = {128, 320, 256, 512, 512, 512};
    const unsigned all = FK_NT_IN | FK_NT_OUT | FK_REAL_QUAD | FK_REAL_UNIT | FK_SWAP_IN;
    int prec, t, i, o, off;
    start();
    for (prec = 0; prec < 2; ++prec)
        for (t = 0; t < 6; ++t)
            for (i = 0; i < 128; i += 4)
                for (o = 0; o < 128; o += 4)
                    for (off = 0; off < 2; ++off) {
                        const long long A = i + (off ? 48 : 0), B = o + (off ? 16 : 0);
                        unsigned w = all;
                        void *buf[FK_NBUF] = {(void *)(0x10000ULL + i), (void *)(0x90000ULL + o)};
                        fk_pass p;
                        fk_args a;
                        memset(&p, 0, sizeof(p));
                        p.k = find_kernel(prec, Ls[t], FK_ROW, ios[t]);
                        p.ibuf = FK_BUF_IN;
                        p.obuf = FK_BUF_OUT;
                        p.ioff = off ? 48 : 0;
                        p.ooff = off ? 16 : 0;
                        p.a.flags = all;
                        fk_bind_pass(&p, buf, &a);
                        if (t < 2 && A % 64) w &= ~FK_NT_IN;
                        if (t < 2 && B % 64) w &= ~FK_NT_OUT;
                        if ((ios[t] == FK_IO_R2C_RR ? A : B) % 16) w &= ~FK_REAL_QUAD;
                        if (ios[t] == FK_IO_DCT4 && (A | B) % (prec ? 8 : 16)) w &= ~FK_REAL_UNIT;
                        CHECK(a.flags == w, "prec=%d io=%d in+%lld out+%lld: flags %u, not %u\n",
                              prec, ios[t], A, B, a.flags, w);
                        CHECK((char *)a.in == (char *)0x10000 + A && (char *)a.out == (char *)0x90000 + B,
                              "addresses\n");
                    }
    printf("%lld %lld\n", bad, seen);
    return 0;
}
""")


def test_first_pass_reads_past_the_caches_by_its_footprint(tmp_path):
    """The first of several FP64 row passes reads non-temporally when its arrays
    exceed the memory-side cache: from 128 MiB each for two arrays, from 384 MiB
    for one that is transformed in place; through staging counts as two."""
    run(tmp_path, EMIT + r"""
int main(void)
{
    const long long MB = 1 << 20;
    int mb, how;
    start();
    for (how = 0; how < 3; ++how) /* out of place, in place, in place into staging */
        for (mb = 64; mb <= 1024; mb += 64) {
            fk_dim b[1] = {{mb * MB / (512 * 16), 512, 512}};
            const int mid = how == 2 ? FK_BUF_S0 : FK_BUF_OUT;
            const unsigned want = mb >= (how == 1 ? 384 : 128) ? FK_NT_IN : 0;
            ctx c;
            fk_plan *P = begin(&c, 0);
            P->inplace = how > 0;
            emit(&c, 0, 512, FK_IO_PLAIN, 1, b, FK_BUF_IN, mid);
            emit(&c, 0, 512, FK_IO_PLAIN, 1, b, mid, FK_BUF_OUT);
            mark_streams(P);
            CHECK((nt(P, 0) & FK_NT_IN) == want && !nt(P, 1), "how=%d %d MiB: %u %u\n", how, mb,
                  nt(P, 0), nt(P, 1));
            free(P->pass);
            free(P);
        }
    printf("%lld %lld\n", bad, seen);
    return 0;
}
""")


def test_rows_in_two_forms_are_taken_by_kind(tmp_path):
    """Where the catalog has a real-to-real row kernel in two forms, the kinds
    that read or write quads take the first (mirrored) by default, the others the
    second; a stored choice is taken as it is."""
    run(tmp_path, r"""
int main(void)
{
    static const int r2c[] = {FK_RM_HC, FK_RM_DHT, FK_RM_E00, FK_RM_O00, FK_RM_DCT2, FK_RM_DST2};
    static const int c2r[] = {FK_RM_HC2R, FK_RM_HC2R, FK_RM_HC2R, FK_RM_HC2R, FK_RM_DCT3, FK_RM_DST3};
    int i, j, v, two = 0;
    start();
    for (i = 0; i < g_nreg; ++i) {
        const fk_kernel *k = g_reg + i, *vs[16];
        int n;
        if (k->variant || k->mode != FK_ROW || (k->io != FK_IO_R2C_RR && k->io != FK_IO_C2R_RR)) continue;
        n = find_variants(k->prec, k->L, k->mode, k->io, vs, 16);
        CHECK(n <= 2, "L=%d: %d forms\n", k->L, n);
        two += n == 2;
        for (j = 0; j < 6; ++j)
            for (v = -1; v < n; ++v) {
                ctx c;
                fk_plan *P = begin(&c, k->prec);
                const int want = v >= 0 ? v : n == 2 && j < 4;
                c.choice = v < 0 ? 0 : &v;
                c.nchoice = v >= 0;
                CHECK(pick_rr_row(&c, k->prec, k->L, k->io, (k->io == FK_IO_R2C_RR ? r2c : c2r)[j]) ==
                          vs[want], "prec=%d L=%d io=%d kind %d choice %d\n", k->prec, k->L, k->io, j, v);
                free(P);
            }
    }
    CHECK(two > 0, "no kernel in two forms\n");
    printf("%lld %lld\n", bad, seen);
    return 0;
}
""")


def test_transposing_lines_without_a_transposed_store(tmp_path):
    """Whole lines strided on one side only: two passes where the length has no
    transposed-store kernel, its split ends in one, the lines of a workgroup make
    short runs and the array is large, the larger the longer the runs are; one pass
    in the other cases, for rows, columns and small batches, and always when scratch
    is to be avoided.  Sizes just below a power of two count as that size."""
    run(tmp_path, r"""
int main(void)
{
    int prec, L, w, taken = 0;
    start();
    for (prec = 0; prec < 2; ++prec)
        for (L = 2; L <= 2048; ++L) {
            const fk_kernel *k = find_kernel(prec, L, FK_ROW, FK_IO_PLAIN);
            long long mb, n1[1];
            int tout = 0;
            if (!k) continue;
            if (!is_factor(prec, L) && split_candidates(prec, L, n1, 1))
                tout = find_kernel(prec, L / n1[0], FK_ROW, FK_IO_TOUT) != 0;
            for (mb = 1; mb <= 256; mb += mb < 32 ? 1 : 16)
                for (w = 0; w < 5; ++w) { /* store, load, rows, columns, store without scratch */
                    const long long H = (mb << 20) / (L * (prec ? 8 : 16)); /* just below */
                    const fk_dim b = {H, w == 1 || w == 3 ? 1 : L, w == 1 || w == 2 ? L : 1};
                    /* the largest size that still is one pass, by lines a workgroup */
                    static const int one_st[2][6] = {{0, 16, 24, 24, 64, 64}, {0, 4, 8, 16, 16, 24}};
                    static const int one_ld[2][6] = {{0, 4}, {0, 4, 4, 4}};
                    static const int two_st[2][6] = {{0, 24, 32, 32, 128, 128}, {0, 8, 12, 24, 24, 32}};
                    const int side = w == 1, q = k->nl > 5 ? 0 : k->nl;
                    const int one = side ? one_ld[prec][q] : one_st[prec][q];
                    const int two = side ? 8 : two_st[prec][q];
                    const int want = tout && w < 2 && one && mb >= two;
                    if (one && mb > one && mb < two) continue; /* either will do */
                    ctx c;
                    fk_plan *P = begin(&c, prec);
                    c.lean = w == 4;
                    CHECK(transposing_split(&c, k, L, w == 1 || w == 3 ? H : 1,
                                            w == 1 || w == 2 ? 1 : H, 1, &b) == want,
                          "prec=%d L=%d nl=%d form %d %lld MiB\n", prec, L, k->nl, w, mb);
                    taken += want;
                    c.lean = 0;
                    c.part = 1;
                    CHECK(!transposing_split(&c, k, L, 1, H, 1, &b), "part of a split\n");
                    free(P);
                }
        }
    CHECK(taken > 100, "only %d\n", taken);
    printf("%lld %lld\n", bad, seen);
    return 0;
}
""")


def test_splits_use_the_lengths_kept_for_them(tmp_path):
    """Every kernel of a length carries the same factor flag, the flagged lengths
    are gen_kernels.factor_list, and the first length of every split candidate
    (up to four per line) is flagged while its rest can be planned from flagged
    lengths."""
    import sys
    sys.path.insert(0, PKG)
    import gen_kernels as g
    lists = "".join("static const int fac_%d[] = {%s, 0};\n" %
                    (i, ",".join(map(str, sorted(g.factor_list(p) & set(g.size_list(p))))))
                    for i, p in ((0, "double"), (1, "float")))
    run(tmp_path, lists + r"""
int main(void)
{
    int prec, i, j, n;
    start();
    for (i = 0; i < g_nreg; ++i) {
        const int *f = g_reg[i].prec ? fac_1 : fac_0;
        int in = 0;
        for (j = 0; f[j]; ++j) in |= f[j] == g_reg[i].L;
        CHECK(in == g_reg[i].factor, "L=%d prec=%d: flag %d\n", g_reg[i].L, g_reg[i].prec, g_reg[i].factor);
    }
    for (prec = 0; prec < 2; ++prec)
        for (n = 2; n < 30000; ++n) {
            long long c[4];
            int nc = smooth_plannable(prec, n, 0) ? split_candidates(prec, n, c, 4) : 0;
            for (j = 0; j < nc; ++j) {
                const fk_kernel *k = find_kernel(prec, c[j], FK_COL, FK_IO_PLAIN);
                CHECK(k && k->factor && smooth_plannable(prec, n / c[j], 1), "n=%d: %lld\n", n, c[j]);
            }
        }
    printf("%lld %lld\n", bad, seen);
    return 0;
}
""")
