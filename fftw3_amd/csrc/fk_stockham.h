/*
 * LDS-resident Stockham kernel: every workgroup transforms NL lines of
 * length L (compile-time L, radix sequence, thread layout).
 *
 * Stage s with radix Rs and Ns = R0*...*R(s-1) (autosort Stockham,
 * decimation in time):
 *   butterfly b in [0, L/Rs), k = b mod Ns
 *   inputs   x[b + r*L/Rs]                        r = 0..Rs-1
 *   twiddle  x_r *= W_{Ns*Rs}^{r*k}
 *   outputs  y[(b/Ns)*Ns*Rs + k + r*Ns] = DFT_Rs(x)_r
 * The first stage reads straight from HBM and the last stage writes straight
 * to HBM (both patterns are unit-stride across threads); the stages between
 * exchange through LDS.  This replaces FFTW's Cooley-Tukey recursion with
 * twiddle codelets (dft/ct.c:34-45, dft/dftw-direct.c:46-56) for every
 * length that fits one workgroup.
 *
 * Line addressing follows FFTW's tensor semantics (kernel/ifftw.h:417-432):
 * element j of line (i0,i1,i2) is at i0*ids0 + i1*ids1 + i2*ids2 + j*is.
 */
#ifndef FK_STOCKHAM_H
#define FK_STOCKHAM_H

#include "fk_device.h"

namespace fk {

template <int... RS>
struct RadList {
    static constexpr int n = sizeof...(RS);
    static constexpr int r[n] = {RS...};
    static constexpr int L()
    {
        int p = 1;
        for (int i = 0; i < n; ++i) p *= r[i];
        return p;
    }
    static constexpr int ns(int s)
    {
        int p = 1;
        for (int i = 0; i < s; ++i) p *= r[i];
        return p;
    }
    /* offset of stage s in the twiddle table (stage 0 has none) */
    static constexpr int twoff(int s)
    {
        int o = 0;
        for (int t = 1; t < s; ++t) o += ns(t) * (r[t] - 1);
        return o;
    }
    static constexpr int twsize() { return twoff(n); }
};

/* Element index b + OFF of a line, b a multiple of ALIGN.  The padded row
   layout keeps the compile-time part OFF out of the per-element address
   arithmetic (it becomes the LDS instruction's offset); every other
   accessor takes the plain index through the conversion. */
template <int OFF, int ALIGN = 1>
struct At {
    int b;
    __device__ __forceinline__ constexpr operator int() const { return b + OFF; }
};

template <class T>
struct AtOff;
template <int OFF, int ALIGN>
struct AtOff<At<OFF, ALIGN>> {
    static constexpr int v = OFF;
};

/* Butterfly I of a thread in a stage of NB butterflies over TPL threads:
   u + I*TPL, or mirrored (needs NB a multiple of 2*TPL): the second half of
   the thread's butterflies are the images b -> NB-1-b of the first, so that
   a thread holds elements j and L-1-j of its line together. */
template <int NB, int TPL, bool MIR>
struct Bfly {
    static constexpr int BPT = (NB + TPL - 1) / TPL;
    static_assert(!MIR || NB % (2 * TPL) == 0, "mirrored mapping");
    template <int I>
    __device__ __forceinline__ static int at(int u)
    {
        if constexpr (MIR && I >= BPT / 2) return NB - 1 - u - (I - BPT / 2) * TPL;
        else return u + I * TPL;
    }
    /* the index of the image of butterfly I */
    static constexpr int image(int I) { return I < BPT / 2 ? I + BPT / 2 : I - BPT / 2; }
};

/* XL = 1 adds one scratch line for threads beyond TPL*NL (a persistent
   workgroup running a geometry smaller than itself). */
template <typename R, int L, int TPL, int NL, int MODE, int PAD, int XL = 0>
struct Geo {
    /* LDS pitch of one line (ROW) — one pad slot every PAD elements, one
       extra slot for the Nyquist bin of the real transforms */
    static constexpr int LP = L + L / PAD + 2;
    static constexpr int NLP = NL + XL;
    __device__ __forceinline__ static int idx(int lt, int j)
    {
        if constexpr (MODE == FK_ROW)
            return lt * LP + j + (int)((unsigned)j / (unsigned)PAD);
        else
            return j * NLP + lt;
    }
    /* (b + OFF) / PAD = b / PAD + OFF / PAD when PAD divides OFF or b */
    template <int OFF, int ALIGN>
    __device__ __forceinline__ static int idx(int lt, At<OFF, ALIGN> j)
    {
        if constexpr (MODE == FK_ROW && (OFF % PAD == 0 || ALIGN % PAD == 0))
            return lt * LP + j.b + (int)((unsigned)j.b / (unsigned)PAD) + (OFF + OFF / PAD);
        else
            return idx(lt, (int)j);
    }
    static constexpr unsigned lds_elems()
    {
        return MODE == FK_ROW ? (unsigned)(NLP * LP) : (unsigned)((L + 2) * NLP);
    }
};

/* Workgroup barrier of the Stockham stages (a policy parameter so that a
   kernel may substitute its own). */
struct SyncAll {
    __device__ __forceinline__ static void sync() { __syncthreads(); }
};

/* Wave-level ordering for stages whose LDS exchange stays inside one wave
   (row mapping with every line's threads in one wave, lines in disjoint
   LDS rows): a wave's LDS accesses complete in issue order, so only the
   compiler must be kept from moving accesses across the exchange point.
   Waves of the workgroup then run their stages independently. */
struct SyncWave {
    __device__ __forceinline__ static void sync()
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
};

/* What happens to a butterfly's registers after its loads (first stage) or
   before its stores (last stage). */
struct NoOp {
    template <int N, int I, typename R>
    __device__ __forceinline__ void run(int, cx<R> *) const
    {
    }
};

/* Swap re and im of N values when the pass runs backward.  The empty asm
   keeps the swap a branch that every wave takes or skips as a whole: as
   selects it would cost the forward direction two instructions a value. */
template <int N, typename R>
__device__ __forceinline__ void swap_if(bool sw, cx<R> *v)
{
    if (sw) {
        asm volatile("");
        sfor<0, N>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            v[r] = swp(v[r]);
        });
    }
}
struct SwapOp {
    bool sw;
    template <int N, int I, typename R>
    __device__ __forceinline__ void run(int, cx<R> *v) const
    {
        swap_if<N>(sw, v);
    }
};

/* Output post-op of the plain passes: four-step twiddle, then the swap.
   The twiddle of output k = b + r*Ns (last stage, r = 0..N-1) of a line with
   batch index i0 is W_N^(k*i0): looked up in the FP64 table every ANCH
   outputs of a butterfly and multiplied by powers of W_N^(Ns*i0) in FP64 in
   between (binary splitting, so that the products do not wait for each
   other).  FP64 data re-anchors every 4 (at most 2 products from a table
   value); FP32 data once per butterfly (at most 4 products, the last power
   itself 3 squarings, ~2e-15, far below FP32 rounding).  The lookups are made
   before the stages, so that they do not add their latency to the end of the
   pass, while they fit a few registers. */
template <typename R, class RL, int TPL>
struct PlainOut {
    static constexpr int N = RL::r[RL::n - 1], NS = RL::ns(RL::n - 1);
    static constexpr int BPT = (NS + TPL - 1) / TPL;
    static constexpr int ANCH = sizeof(R) == 8 ? 4 : 16, NA = (N + ANCH - 1) / ANCH;
    static constexpr bool EARLY = sizeof(R) == 4 && BPT * NA <= 4;
    const fk_args &a;
    bool tw, sw;
    long long i0;
    cx<double> step, anchor[EARLY ? BPT * NA : 1];
    __device__ __forceinline__ PlainOut(const fk_args &a_, unsigned fl, long long i0_, int u)
        : a(a_), tw(fl & FK_TW_OUT), sw(fl & FK_SWAP_OUT), i0(i0_), step(mk(1.0, 0.0))
    {
        if (tw) {
            step = tw2d(a, (long long)NS * i0);
            if constexpr (EARLY)
                sfor<0, BPT * NA>([&](auto ic) {
                    constexpr int i = decltype(ic)::value / NA, g = decltype(ic)::value % NA;
                    /* threads past the last butterfly look up the last one's */
                    const int b = u + i * TPL < NS ? u + i * TPL : NS - 1;
                    anchor[i * NA + g] = tw2d(a, (long long)(b + g * ANCH * NS) * i0);
                });
        }
    }
    template <int N_, int I>
    __device__ __forceinline__ void run(int b, cx<R> *v) const
    {
        if (tw) {
            const cx<double> s2 = mul(step, step);
            cx<double> s4 = s2, s8 = s2;
            if constexpr (ANCH > 4 && N > 4) s4 = mul(s2, s2);
            if constexpr (ANCH > 8 && N > 8) s8 = mul(s4, s4);
            sfor<0, NA>([&](auto gc) {
                constexpr int g = decltype(gc)::value;
                cx<double> w[ANCH];
                if constexpr (EARLY) w[0] = anchor[I * NA + g];
                else w[0] = tw2d(a, (long long)(b + g * ANCH * NS) * i0);
                sfor<1, ANCH>([&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    constexpr int h = r >= 8 ? 8 : r >= 4 ? 4 : r >= 2 ? 2 : 1;
                    if constexpr (g * ANCH + r < N)
                        w[r] = mul(w[r - h], h == 8 ? s8 : h == 4 ? s4 : h == 2 ? s2 : step);
                });
                sfor<0, ANCH>([&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    if constexpr (g * ANCH + r < N)
                        v[g * ANCH + r] = mul(v[g * ANCH + r], mk((R)w[r].x, (R)w[r].y));
                });
            });
        }
        swap_if<N>(sw, v);
    }
};

/*
 * One Stockham stage.  LoadF(j) -> cx<R> and StoreF(k, cx<R>) abstract the
 * data source and sink (or are Hoisted); IN_LDS/OUT_LDS say whether they
 * touch LDS, which decides the barriers.  pre / fin run on a butterfly's registers after the
 * loads / before the stores.
 */
template <typename R, class RL, int S, int L, int TPL, bool IN_LDS, bool OUT_LDS, bool MIR,
          class SY, class LoadF, class StoreF, class PreF, class FinF>
__device__ __forceinline__ void stage(int u, const cx<R> *__restrict__ tw,
                                      LoadF &&ld, StoreF &&st, const PreF &pre, const FinF &fin)
{
    constexpr int Rs = RL::r[S];
    constexpr int Ns = RL::ns(S);
    constexpr int NB = L / Rs;
    using BF = Bfly<NB, TPL, MIR>;
    constexpr int BPT = BF::BPT;
    cx<R> v[BPT][Rs];
    auto load = [&](auto &&get) {
        sfor<0, BPT>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const int b = BF::template at<i>(u);
            if ((NB % TPL == 0) || b < NB) {
                sfor<0, Rs>([&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    v[i][r] = get(At<r * NB>{b});
                });
            }
        });
    };
    typedef typename std::decay<LoadF>::type Ld;
    typedef typename std::decay<StoreF>::type St;
    if constexpr (is_whole<Ld>::value) ld.f(v);
    else if constexpr (is_hoisted<Ld>::value) ld.f(load);
    else load(ld);
    if constexpr (IN_LDS && OUT_LDS) SY::sync();
    sfor<0, BPT>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const int b = BF::template at<i>(u);
        if ((NB % TPL == 0) || b < NB) {
            /* the last stage has Ns = NB, so b < Ns there: its outputs are
               b + r*Ns, a compile-time offset from the thread's index */
            const int k = S == RL::n - 1 ? b : b % Ns;
            if constexpr (S > 0) {
                const cx<R> *w = tw + RL::twoff(S) + k * (Rs - 1);
                sfor<1, Rs>([&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    v[i][r] = mul(v[i][r], w[r - 1]);
                });
            }
            pre.template run<Rs, i>(b, v[i]);
            Dft<R, Rs, 1>::run(v[i]);
            const int base = (b - k) * Rs + k;
            fin.template run<Rs, i>(base, v[i]);
            /* stage 0 (Ns = 1) writes Rs consecutive outputs from b*Rs */
            auto store = [&](auto &&put) {
                sfor<0, Rs>([&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    put(At<r * Ns, (S == 0 ? Rs : 1)>{base}, v[i][r]);
                });
            };
            if constexpr (is_hoisted<St>::value) st.f(store);
            else if constexpr (!is_whole<St>::value) store(st);
        }
    });
    if constexpr (is_whole<St>::value) st.f(v);
    if constexpr (OUT_LDS) SY::sync();
}

/* Runs stages [S, RL::n) ; stage S loads with `first` (then `pre`), the last
   stage stores with `last` (after `fin`), everything between goes through
   LDS.  M0 / ML: mirrored mapping of the first / last stage. */
template <typename R, class RL, int S, int L, int TPL, bool FIRST_LDS,
          bool LAST_LDS, class SY = SyncAll, bool M0 = false, bool ML = false, class LdsF,
          class FirstF, class LastF, class PreF = NoOp, class FinF = NoOp>
__device__ __forceinline__ void run_stages(int u, const cx<R> *tw, LdsF &&lds,
                                           FirstF &&first, LastF &&last,
                                           const PreF &pre = PreF(), const FinF &fin = FinF())
{
    constexpr int n = RL::n;
    auto lds_ld = [&](auto j) { return lds(j); };
    auto lds_st = [&](auto k, cx<R> v) { lds(k) = v; };
    if constexpr (S == 0 && n == 1) {
        static_assert(!M0 && !ML, "one-stage kernels are not mirrored");
        stage<R, RL, 0, L, TPL, FIRST_LDS, LAST_LDS, false, SY>(u, tw, first, last, pre, fin);
    } else if constexpr (S == 0) {
        stage<R, RL, 0, L, TPL, FIRST_LDS, true, M0, SY>(u, tw, first, lds_st, pre, NoOp());
        run_stages<R, RL, 1, L, TPL, FIRST_LDS, LAST_LDS, SY, M0, ML>(u, tw, lds, first, last, NoOp(),
                                                                     fin);
    } else if constexpr (S == n - 1) {
        stage<R, RL, S, L, TPL, true, LAST_LDS, ML, SY>(u, tw, lds_ld, last, NoOp(), fin);
    } else {
        stage<R, RL, S, L, TPL, true, true, false, SY>(u, tw, lds_ld, lds_st, NoOp(), NoOp());
        run_stages<R, RL, S + 1, L, TPL, FIRST_LDS, LAST_LDS, SY, M0, ML>(u, tw, lds, first, last,
                                                                         NoOp(), fin);
    }
}

/* whether the first / last stage of a kernel can run mirrored with whole
   element pairs: an even radix and a multiple of 2*TPL butterflies */
template <class RL, int TPL>
struct MirOk {
    static constexpr int L = RL::L(), R0 = RL::r[0], RN = RL::r[RL::n - 1];
    /* one thread holds the whole line: every element's image is its own */
    static constexpr bool self = RL::n == 1 && TPL == 1 && R0 % 2 == 0;
    static constexpr bool first = RL::n > 1 && R0 % 2 == 0 && (L / R0) % (2 * TPL) == 0;
    static constexpr bool last = RL::n > 1 && RN % 2 == 0 && (L / RN) % (2 * TPL) == 0;
};

__device__ __forceinline__ long long remap_tile(unsigned xcd)
{
    const unsigned w = blockIdx.x;
    if (!xcd) return w;
    /* workgroups are dispatched round-robin over 8 XCDs; give each XCD a
       contiguous run of tiles so neighbouring tiles share its L2 */
    const unsigned nwg = gridDim.x, per = nwg / 8, rem = nwg % 8;
    const unsigned x = w % 8, i = w / 8;
    return x * per + (x < rem ? x : rem) + i;
}

/*
 * Body of one workgroup tile: lines [tile*NL, tile*NL + NL).  NT is the
 * workgroup size; when NT > TPL*NL (persistent workgroups shared by several
 * geometries) the extra threads work on a scratch LDS line and never touch
 * global memory, so every thread still meets every barrier.
 */
template <typename R, int NL, int MODE, int IO, int PAD, class RL, int TPL, int NT,
          class SY = SyncAll>
__device__ __forceinline__ void stockham_body(const fk_args &a, long long tile,
                                              unsigned char *smem_raw)
{
    constexpr int L = RL::L();
    constexpr int NR = TPL * NL;
    using G = Geo<R, L, TPL, NL, MODE, PAD>;
    static_assert(NT >= NR, "workgroup smaller than the geometry");
    cx<R> *lds = reinterpret_cast<cx<R> *>(smem_raw);
    long long *lbase = reinterpret_cast<long long *>(lds + G::lds_elems());
    /* threads beyond TPL*NL read and write a 64-slot trash area */
    cx<R> *trash = reinterpret_cast<cx<R> *>(lbase + ((NL + 1) & ~1));

    const int tid = threadIdx.x;
    const bool real = (NT == NR) || tid < NR;
    /* row mapping with whole waves per line: the line, and all that follows
       from it, is computed once per wave on the scalar unit */
    constexpr bool UNI = MODE == FK_ROW && TPL % 64 == 0;
    const int lt_ = !real ? 0 : (MODE == FK_ROW) ? tid / TPL : tid % NL;
    const int lt = UNI ? __builtin_amdgcn_readfirstlane(lt_) : lt_;
    const int u = !real ? (tid - NR) % TPL : (MODE == FK_ROW) ? tid % TPL : tid / NL;
    const long long line = tile * NL + lt;
    const bool act = real && line < a.nlines;

    /* inactive lanes take line 0 (in bounds) */
    const LineIx lx = line_ix(a, act ? line : 0);
    const long long i0 = lx.i0;
    long long bin, bout;
    line_off(a, lx, bin, bout);
    const cx<R> *tw = reinterpret_cast<const cx<R> *>(a.tw);
    const unsigned fl = a.flags;
    const bool swi = fl & FK_SWAP_IN, swo = fl & FK_SWAP_OUT;
    const bool nti = fl & FK_NT_IN, nto = fl & FK_NT_OUT;
    /* kernels that the non-temporal flags can reach (whole_sectors in engine.c) */
    constexpr int NB_0 = L / RL::r[0], NB_N = L / RL::r[RL::n - 1];
    constexpr bool NTP = sizeof(R) == 8 && MODE == FK_ROW && IO == FK_IO_PLAIN && TPL % 4 == 0 &&
                         NB_0 % 4 == 0 && NB_N % 4 == 0;
    auto lds_at = [&](auto j) -> cx<R> & {
        if constexpr (NT == NR) return lds[G::idx(lt, j)];
        else return real ? lds[G::idx(lt, j)] : trash[tid & 63];
    };

    if constexpr (IO == FK_IO_PLAIN || IO == FK_IO_TOUT) {
        /* element j of the thread's line sits (j - u) strides from the
           thread's own element u; the stages pass j = u + (compile-time
           offset), so each access is one uniform product and one 64-bit
           add.  Inactive lanes read line 0 (in bounds) and store nothing. */
        const long long is = a.is, os = a.os;
        const cx<R> *inu = reinterpret_cast<const cx<R> *>(a.in) + bin + u * is;
        cx<R> *out = reinterpret_cast<cx<R> *>(a.out);
        auto gld = hoisted([&](auto &&load) {
            with_acc(NTP && nti, [&](auto acc) {
                load([&](int j) -> cx<R> { return ldg(acc, inu + (long long)(j - u) * is); });
            });
        });
        if constexpr (IO == FK_IO_PLAIN) {
            cx<R> *outu = out + bout + u * os;
            auto gst = hoisted([&](auto &&store) {
                with_acc(NTP && nto, [&](auto acc) {
                    store([&](int k, cx<R> v) {
                        if (act) stg(acc, outu + (long long)(k - u) * os, v);
                    });
                });
            });
            const PlainOut<R, RL, TPL> fin(a, fl, i0, u);
            run_stages<R, RL, 0, L, TPL, false, false, SY>(u, tw, lds_at, gld, gst, SwapOp{swi},
                                                           fin);
        } else {
            auto lst = [&](auto k, cx<R> v) { lds_at(k) = v; };
            /* output offsets may be negative (negative strides): inactive
               lines are marked with the one value no offset takes */
            constexpr long long NONE = -0x7fffffffffffffffLL - 1; /* INT64_MIN */
            if (u == 0 && real) lbase[lt] = act ? bout : NONE;
            run_stages<R, RL, 0, L, TPL, false, true, SY>(u, tw, lds_at, gld, lst, SwapOp{swi},
                                                          SwapOp{swo});
            /* the store below reads every line of the tile */
            if constexpr (!std::is_same<SY, SyncAll>::value) __syncthreads();
            /* lines-fastest store: consecutive threads write consecutive
               lines of the tile (unit output batch stride) */
            for (int e = tid; e < NL * L; e += NT) {
                const int l2 = e % NL, k = e / NL;
                const long long ob = lbase[l2];
                if (ob != NONE) out[ob + k * a.os] = lds[G::idx(l2, k)];
            }
        }
    } else if constexpr (IO == FK_IO_R2C_FULL) {
        /* r2c of a length-L real line whose half length has no kernel (odd
           L): the full L-point DFT of (x_j, 0); bins k <= L/2 are stored */
        const R *inr = reinterpret_cast<const R *>(a.in) + bin;
        cx<R> *out = reinterpret_cast<cx<R> *>(a.out);
        auto gld = [&](int j) -> cx<R> {
            return act ? mk(inr[(long long)j * a.is], (R)0) : mk((R)0, (R)0);
        };
        auto gst = [&](int k, cx<R> v) {
            if (act && 2 * k <= L) out[bout + (long long)k * a.os] = v;
        };
        run_stages<R, RL, 0, L, TPL, false, false, SY>(u, tw, lds_at, gld, gst);
    } else if constexpr (IO == FK_IO_C2R_FULL) {
        /* c2r of length L from bins k <= L/2: X_{L-k} = conj X_k (Im X_0 and,
           for even L, Im X_{L/2} ignored); the inverse DFT as a forward DFT
           of swap(X), whose real output part is Im of the result */
        const cx<R> *in = reinterpret_cast<const cx<R> *>(a.in) + bin;
        R *outr = reinterpret_cast<R *>(a.out) + bout;
        auto gld = [&](int j) -> cx<R> {
            if (!act) return mk((R)0, (R)0);
            cx<R> v;
            if (2 * j <= L) {
                v = in[(long long)j * a.is];
                if (j == 0 || 2 * j == L) v.y = (R)0;
            } else {
                v = in[(long long)(L - j) * a.is];
                v.y = -v.y;
            }
            return swp(v);
        };
        auto gst = [&](int k, cx<R> v) {
            if (act) outr[(long long)k * a.os] = v.y;
        };
        run_stages<R, RL, 0, L, TPL, false, false, SY>(u, tw, lds_at, gld, gst);
    } else if constexpr (IO == FK_IO_DCT4) {
        /* REDFT11 of n = 2L reals: z_m = (x_2m + i x_{n-1-2m}) exp(-i pi (4m+1) / 4n),
           Z = L-point DFT, c_p = Z_p exp(-i pi p / n), y_2p = 2 Re c_p,
           y_{n-1-2p} = -2 Im c_p.  RODFT11_k(x) = (-1)^k REDFT11_k(x reversed).
           rtw holds the L input twiddles, then the L output twiddles.  The
           sine kind's z_m is the cosine kind's with re and im swapped.  With
           the mirrored mapping a thread has elements m and L-1-m, samples 2m,
           2m+1 and n-2-2m, n-1-2m of the line on both sides: pairs of
           neighbours (FK_REAL_UNIT: unit strides, pairs aligned). */
        const R *inr = reinterpret_cast<const R *>(a.in) + bin;
        R *outr = reinterpret_cast<R *>(a.out) + bout;
        const cx<R> *t0 = reinterpret_cast<const cx<R> *>(a.rtw), *t1 = t0 + L;
        const bool sn = a.rmode == FK_RM_DST4;
        const long long is = a.is, os = a.os;
        constexpr long long N2 = 2LL * L;
        constexpr int R0 = RL::r[0], NB0 = L / R0, RN = RL::r[RL::n - 1], NBN = L / RN;
        constexpr bool M0 = MirOk<RL, TPL>::first, ML = MirOk<RL, TPL>::last;
        constexpr bool SELF = MirOk<RL, TPL>::self;
        using BF0 = Bfly<NB0, TPL, M0>;
        using BFN = Bfly<NBN, TPL, ML>;
        auto first = whole([&](auto &v) {
            if ((M0 || SELF) && (fl & FK_REAL_UNIT)) {
                asm volatile("");
                if constexpr (SELF) {
                    const cx<R> *p = reinterpret_cast<const cx<R> *>(inr);
                    cx<R> x[R0];
                    sfor<0, R0>([&](auto rc) { x[decltype(rc)::value] = p[decltype(rc)::value]; });
                    sfor<0, R0>([&](auto rc) {
                        constexpr int r = decltype(rc)::value;
                        v[0][r] = mk(x[r].x, x[R0 - 1 - r].y);
                    });
                } else if constexpr (M0)
                    sfor<0, BF0::BPT / 2>([&](auto ic) {
                        constexpr int i = decltype(ic)::value, im = BF0::image(i);
                        const cx<R> *p = reinterpret_cast<const cx<R> *>(inr);
                        const cx<R> *pi = p + BF0::template at<i>(u), *pm = p + BF0::template at<im>(u);
                        cx<R> x[R0], y[R0];
                        sfor<0, R0>([&](auto rc) {
                            constexpr int r = decltype(rc)::value;
                            x[r] = ldg(Acc<C_ONCE>{}, pi + r * NB0);
                            y[r] = ldg(Acc<C_ONCE>{}, pm + r * NB0);
                        });
                        sfor<0, R0>([&](auto rc) {
                            constexpr int r = decltype(rc)::value;
                            v[i][r] = mk(x[r].x, y[R0 - 1 - r].y);
                            v[im][r] = mk(y[r].x, x[R0 - 1 - r].y);
                        });
                    });
            } else {
                sfor<0, BF0::BPT>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    const int b = BF0::template at<i>(u);
                    if ((NB0 % TPL == 0) || b < NB0) {
                        const R *p = inr + 2 * b * is, *q = inr + (N2 - 1 - 2 * b) * is;
                        sfor<0, R0>([&](auto rc) {
                            constexpr int r = decltype(rc)::value;
                            const long long o = (2LL * r * NB0) * is;
                            v[i][r] = mk(p[o], q[-o]);
                        });
                    }
                });
            }
            sfor<0, BF0::BPT>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                const int b = BF0::template at<i>(u);
                if ((NB0 % TPL == 0) || b < NB0) {
                    swap_if<R0>(sn, v[i]);
                    sfor<0, R0>([&](auto rc) {
                        constexpr int r = decltype(rc)::value;
                        v[i][r] = mul(v[i][r], t0[b + r * NB0]);
                    });
                }
            });
        });
        auto last = whole([&](auto &v) {
            sfor<0, BFN::BPT>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                const int b = BFN::template at<i>(u);
                if ((NBN % TPL == 0) || b < NBN)
                    sfor<0, RN>([&](auto rc) {
                        constexpr int r = decltype(rc)::value;
                        const cx<R> c = mul(v[i][r], t1[b + r * NBN]);
                        const R yo = (R)-2 * c.y;
                        v[i][r] = mk((R)2 * c.x, sn ? -yo : yo);
                    });
            });
            sfor<0, BFN::BPT>([&](auto ic) {
                constexpr int i = decltype(ic)::value, im = ML ? BFN::image(i) : i;
                const int b = BFN::template at<i>(u);
                if (act && ((NBN % TPL == 0) || b < NBN)) {
                    if ((ML || SELF) && (fl & FK_REAL_UNIT)) {
                        asm volatile("");
                        cx<R> *p = reinterpret_cast<cx<R> *>(outr) + b;
                        sfor<0, RN>([&](auto rc) {
                            constexpr int r = decltype(rc)::value;
                            p[r * NBN] = mk(v[i][r].x, v[im][RN - 1 - r].y);
                        });
                    } else {
                        R *p = outr + 2 * b * os, *q = outr + (N2 - 1 - 2 * b) * os;
                        sfor<0, RN>([&](auto rc) {
                            constexpr int r = decltype(rc)::value;
                            const long long o = (2LL * r * NBN) * os;
                            p[o] = v[i][r].x;
                            q[-o] = v[i][r].y;
                        });
                    }
                }
            });
        });
        run_stages<R, RL, 0, L, TPL, false, false, SY, M0, ML>(u, tw, lds_at, first, last);
    } else if constexpr (IO == FK_IO_R2C || IO == FK_IO_R2C_XR) {
        /* real line of 2L samples viewed as L complex z_j = x_2j + i x_2j+1;
           after the L-point DFT Z, X[k] = E[k] + W_2L^k O[k] with
           E = (Z[k] + conj Z[L-k])/2, O = (Z[k] - conj Z[L-k])/(2i),
           k = 0..L (the role of rdft/ct-hc2c.c:197-210's HC2C_VIA_DFT).
           What bounds it: the twiddle loads of its three stages and of the
           post-pass outnumber the data loads and live in the CU's L1, which
           the data streams through.  Data read past L1 (C_ONCE) leaves the
           tables there: FP32 2048 x 65536 0.246 -> 0.205 ms.  Not where few
           threads read a line: a sector that several loads share is then
           fetched by each of them (64 MiB of FP32 input, us cached / C_ONCE:
           14 samples, 1 thread, 58 / 69; 52, 2 threads, 47 / 60; 36, 3 threads,
           46 / 50; 84, 6 threads, 45 / 39; with 4 threads only lines that start
           at a sector: 64 samples 53 / 41, 56 samples 42 / 45). */
        constexpr int ONCE = TPL >= 6 || (TPL == 4 && L % 8 == 0) ? C_ONCE : C_KEEP;
        const R *inr = reinterpret_cast<const R *>(a.in) + bin;
        cx<R> *out = reinterpret_cast<cx<R> *>(a.out);
        const cx<R> *wk = reinterpret_cast<const cx<R> *>(a.aux);
        const long long is = a.is, os = a.os;
        auto gld = hoisted([&](auto &&load) {
            if (fl & FK_REAL_UNIT) {
                const cx<R> *inz = reinterpret_cast<const cx<R> *>(inr) + u;
                load([&](int j) -> cx<R> { return ldg(Acc<ONCE>{}, inz + (j - u)); });
            } else {
                asm volatile("");
                const R *inu = inr + 2 * u * is;
                load([&](int j) -> cx<R> {
                    const long long o = 2 * (j - u) * is;
                    return mk(inu[o], inu[o + is]);
                });
            }
        });
        auto lst = [&](auto k, cx<R> v) { lds_at(k) = v; };
        /* bin k <= L/2 gives bins k and L-k from the same Z[k], Z[L-k] and
           one twiddle (W_2L^(L-k) = -conj W_2L^k); bins k = u + i*TPL in
           groups of 8 (compile-time count): the group's twiddle loads are
           in flight together */
        constexpr int HK = L / 2;
        constexpr int NK2 = (HK + 1 + TPL - 1) / TPL;
        constexpr int GK = 8;
        constexpr bool XR = IO == FK_IO_R2C_XR;
        /* few bins per thread: their twiddles are loaded before the stages,
           so the load latency hides behind the FFT instead of following it */
        constexpr bool PRE = NK2 <= 20;
        cx<R> wpre[PRE ? NK2 : 1];
        if constexpr (PRE) {
            sfor<0, NK2>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                const int k = u + i * TPL;
                wpre[i] = wk[k <= HK ? k : HK];
            });
        }
        /* cross-row form: twiddles of the first column stage, W_n0^(n1*p) (n1 =
           the tile's line-group index, uniform over the workgroup).  Below 1024
           points they are looked up before the stages, whose loads hide the
           lookups (r2c of 1024 x 1024 x 64 FP32 231 us after them, 208 before,
           x 32 FP64 199 / 190); at 1024, where they cost 12 registers, after
           (2048 x 2048 x 64 FP32 890.6, before 892.8) */
        long long tin = 0, tout = 0;
        cx<R> wp[XR ? NL : 1];
        auto column_tw = [&]() {
            const LineIx tx = line_ix(a, tile * NL);
            line_off(a, tx, tin, tout);
            sfor<0, NL>([&](auto pc) {
                constexpr int pp = decltype(pc)::value;
                wp[pp] = pp == 0 ? mk((R)1, (R)0) : tw2<R>(a, tx.i1 * pp);
            });
        };
        if constexpr (XR && L < 1024) column_tw();
        run_stages<R, RL, 0, L, TPL, false, true, SY>(u, tw, lds_at, gld, lst);
        /* bins k = u + i*TPL <= L/2 and L-k of the line: f(i, k, X[k], X[L-k]) */
        auto bins = [&](auto &&f) {
            sfor<0, (NK2 + GK - 1) / GK>([&](auto gc) {
                constexpr int g = decltype(gc)::value;
                constexpr int cnt = (NK2 - g * GK) < GK ? (NK2 - g * GK) : GK;
                cx<R> w[cnt];
                sfor<0, cnt>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    const int k = u + (g * GK + i) * TPL;
                    if constexpr (PRE) w[i] = wpre[g * GK + i];
                    else if (k <= HK) w[i] = wk[k];
                });
                sfor<0, cnt>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    const int k = u + (g * GK + i) * TPL;
                    if (k <= HK) {
                        const cx<R> zk = lds_at(k);
                        const cx<R> zc = lds_at(k == 0 ? 0 : L - k);
                        const R er = (R)0.5 * (zk.x + zc.x), ei = (R)0.5 * (zk.y - zc.y);
                        /* O = (Z[k] - conj Z[L-k]) / (2i) */
                        const R orr = (R)0.5 * (zk.y + zc.y), oi = (R)-0.5 * (zk.x - zc.x);
                        const R wx = w[i].x, wy = w[i].y;
                        /* X[k] = E + W O; X[L-k] = conj(E - W O), written as
                           the form of bin L-k on its own (E' = conj E,
                           O' = conj O, W' = -conj W) so that both round as
                           that form does */
                        const cx<R> X = mk(er + orr * wx - oi * wy, ei + orr * wy + oi * wx);
                        const cx<R> Y =
                            mk(er + orr * (-wx) - (-oi) * wy, (-ei) + orr * wy + (-oi) * (-wx));
                        f(std::integral_constant<int, g * GK + i>{}, k, X, Y);
                    }
                });
            });
        };
        if constexpr (!XR) {
            cx<R> *outk = out + bout + u * os, *outm = out + bout + (L - u) * os;
            bins([&](auto ic, int k, cx<R> X, cx<R> Y) {
                const long long d = (long long)(decltype(ic)::value * TPL) * os;
                if (act) {
                    outk[d] = X;
                    if (2 * k != L) outm[-d] = Y;
                }
            });
        } else {
            if constexpr (L >= 1024) column_tw();
            /* the bins stay in registers until every bin of the line has
               been formed, then replace Z in the line's LDS row */
            cx<R> xs[2 * NK2];
            bins([&](auto ic, int, cx<R> X, cx<R> Y) {
                constexpr int i = decltype(ic)::value;
                xs[2 * i] = X;
                xs[2 * i + 1] = Y;
            });
            SY::sync();
            sfor<0, NK2>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                const int k = u + i * TPL;
                if (k <= HK) {
                    lds_at(k) = xs[2 * i];
                    if (2 * k != L) lds_at(L - k) = xs[2 * i + 1];
                }
            });
            __syncthreads();
            /* first stage of the column DFT over the tile's NL rows
               n = n1 + m*n2 (n2 = the line's batch index i0, n1 = i1; the
               planner sets nb[0] = NL, so a tile is one n1 and always whole):
               for every bin k y_p = W_n0^(n1*p) sum_n2 X_n2[k] W_NL^(n2*p),
               n0 = a.tN, stored to the tile's output line p */
            cx<R> *outk = out + tout + tid * os;
            for (int k = tid; k <= L; k += NT, outk += NT * os) {
                cx<R> v[NL];
                sfor<0, NL>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    v[q] = lds[G::idx(q, k)];
                });
                Dft<R, NL, 1>::run(v);
                sfor<0, NL>([&](auto pc) {
                    constexpr int pp = decltype(pc)::value;
                    outk[pp * a.ods[0]] = pp == 0 ? v[0] : mul(v[pp], wp[pp]);
                });
            }
        }
    } else if constexpr (IO == FK_IO_C2R || IO == FK_IO_C2R_XR) {
        /* half-length inverse: Z[k] = E[k] + i O[k],
           E[k] = X[k] + conj X[L-k], O[k] = (X[k] - conj X[L-k]) W_2L^-k,
           z = DFT^-1_L(Z) (unnormalized), y_2m = Re z_m, y_2m+1 = Im z_m.
           Im X[0] and Im X[L] are ignored, as the r2cb codelets do. */
        const cx<R> *in = reinterpret_cast<const cx<R> *>(a.in);
        R *outr = reinterpret_cast<R *>(a.out) + bout;
        const cx<R> *wk = reinterpret_cast<const cx<R> *>(a.aux);
        const long long is = a.is, os = a.os;
        /* bins X[k], X[L-k] (k <= L/2) are read together and give Z[k] and
           Z[L-k] with one twiddle (W_2L^(L-k) = -conj W_2L^k); they are
           written to LDS before the stages, which read Z as it is */
        constexpr int HK = L / 2;
        constexpr int NK2 = (HK + 1 + TPL - 1) / TPL;
        constexpr int GK = 8;
        /* swapped Z (the backward DFT runs as the forward one on swapped
           data): e = X[k] + conj X[L-k], d = X[k] - conj X[L-k],
           o = d conj(W_2L^k); Z[k] = e + i o and, by the symmetry above,
           Z[L-k] = conj e + i conj o */
        auto zpair = [&](int k, cx<R> xk, cx<R> xc, cx<R> w, cx<R> &z0, cx<R> &z1) {
            if (k == 0) {
                xk.y = 0;
                xc.y = 0;
            }
            const cx<R> e = mk(xk.x + xc.x, xk.y - xc.y);
            const cx<R> d = mk(xk.x - xc.x, xk.y + xc.y);
            const cx<R> o = mk(d.x * w.x + d.y * w.y, d.y * w.x - d.x * w.y);
            z0 = mk(e.y + o.x, e.x - o.y);
            z1 = mk(o.x - e.y, e.x + o.y);
        };
        if constexpr (IO == FK_IO_C2R_XR) {
            /* last stage of the inverse column DFT over the tile's NL input
               rows (row p = the line's batch index i0, n1 = i1; the planner
               sets nb[0] = NL, so a tile is one n1 and always whole): for
               every bin k u_n2 = sum_p W_NL^(-n2*p) W_n0^(-n1*p) Y_p[k],
               n0 = a.tN, which is line n2's half spectrum (its own output
               row); the inverse DFT as the forward one on swapped data. */
            const LineIx tx = line_ix(a, tile * NL);
            long long tin, tout;
            line_off(a, tx, tin, tout);
            cx<R> wp[NL];
            sfor<0, NL>([&](auto pc) {
                constexpr int pp = decltype(pc)::value;
                const cx<R> t = pp == 0 ? mk((R)1, (R)0) : tw2<R>(a, tx.i1 * pp);
                wp[pp] = mk(t.x, -t.y);
            });
            auto coldft = [&](cx<R> *v) {
                sfor<0, NL>([&](auto pc) {
                    constexpr int pp = decltype(pc)::value;
                    v[pp] = swp(pp == 0 ? v[0] : mul(v[pp], wp[pp]));
                });
                Dft<R, NL, 1>::run(v);
            };
            auto put = [&](int k, cx<R> w, cx<R> *v, cx<R> *vm) {
                sfor<0, NL>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    cx<R> z0, z1;
                    zpair(k, swp(v[q]), swp(vm[q]), w, z0, z1);
                    lds[G::idx(q, k)] = z0;
                    if (k != 0 && 2 * k != L) lds[G::idx(q, L - k)] = z1;
                });
            };
            const cx<R> *ink = in + tin + tid * is, *inm = in + tin + (L - tid) * is;
            auto fetch = [&](const cx<R> *p, cx<R> *v) {
                sfor<0, NL>([&](auto pc) {
                    constexpr int pp = decltype(pc)::value;
                    v[pp] = ldg(Acc<C_ONCE>{}, p + pp * a.ids[0]);
                });
            };
            if constexpr (HK % NT == 0) {
                /* bin L/2 is thread 0's as well: its loads are issued with the
                   others', so that no wave waits for memory twice */
                cx<R> vh[NL];
                if (tid == 0) fetch(in + tin + HK * is, vh);
                for (int k = tid; k < HK; k += NT, ink += NT * is, inm -= NT * is) {
                    cx<R> v[NL], vm[NL];
                    fetch(ink, v);
                    fetch(inm, vm);
                    const cx<R> w = wk[k];
                    coldft(v);
                    coldft(vm);
                    put(k, w, v, vm);
                }
                if (tid == 0) {
                    coldft(vh);
                    put(HK, wk[HK], vh, vh);
                }
            } else {
                /* a thread of its own for bin L/2: one bin pair after the other
                   takes fewer registers (512 points, VGPRs 100 instead of 162 in
                   FP64, 56 instead of 101 in FP32: twice / 1.5 times the
                   workgroups a CU; c2r of 1024 x 1024 x 32 FP64 218 -> 200 us, x
                   64 FP32 221 -> 206) */
                for (int k = tid; k <= HK; k += NT) {
                    const cx<R> w = wk[k];
                    cx<R> v[NL], vm[NL];
                    fetch(in + tin + k * is, v);
                    coldft(v);
                    if (2 * k != L) {
                        fetch(in + tin + (L - k) * is, vm);
                        coldft(vm);
                    }
                    sfor<0, NL>([&](auto qc) {
                        constexpr int q = decltype(qc)::value;
                        const cx<R> xk = swp(v[q]), xc = 2 * k == L ? xk : swp(vm[q]);
                        cx<R> z0, z1;
                        zpair(k, xk, xc, w, z0, z1);
                        lds[G::idx(q, k)] = z0;
                        if (k != 0 && 2 * k != L) lds[G::idx(q, L - k)] = z1;
                    });
                }
            }
            __syncthreads();
        } else {
            /* loads in groups of 8 (compile-time count) so that each group
               is in flight at once, then its LDS stores; through L1, since
               the bins k and L-k of short lines share sectors (64 MiB of FP32
               output, us with C_ONCE / this: 30 samples 49.6 / 39.6, 64 41.1 /
               32.1, 128 33.4 / 28.2, 320 36.7 / 33.2; from 512 on the same) */
            const cx<R> *ink = in + bin + u * is, *inm = in + bin + (L - u) * is;
            sfor<0, (NK2 + GK - 1) / GK>([&](auto gc) {
                constexpr int g = decltype(gc)::value;
                constexpr int cnt = (NK2 - g * GK) < GK ? (NK2 - g * GK) : GK;
                cx<R> xa[cnt], xb[cnt], w[cnt];
                sfor<0, cnt>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    const int k = u + (g * GK + i) * TPL;
                    const long long d = (long long)((g * GK + i) * TPL) * is;
                    if (k <= HK) {
                        xa[i] = ink[d];
                        xb[i] = inm[-d];
                        w[i] = wk[k];
                    }
                });
                sfor<0, cnt>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    const int k = u + (g * GK + i) * TPL;
                    if (k <= HK) {
                        cx<R> z0, z1;
                        zpair(k, xa[i], xb[i], w[i], z0, z1);
                        lds_at(k) = z0;
                        if (k != 0 && 2 * k != L) lds_at(L - k) = z1;
                    }
                });
            });
            SY::sync();
        }
        auto gst = hoisted([&](auto &&store) {
            /* v = swap(z_k) */
            if (fl & FK_REAL_UNIT) {
                cx<R> *outz = reinterpret_cast<cx<R> *>(outr) + u;
                store([&](int k, cx<R> v) {
                    if (act) outz[k - u] = mk(v.y, v.x);
                });
            } else {
                asm volatile("");
                R *outu = outr + 2 * u * os;
                store([&](int k, cx<R> v) {
                    const long long o = 2 * (k - u) * os;
                    if (act) {
                        outu[o] = v.y;
                        outu[o + os] = v.x;
                    }
                });
            }
        });
        auto zld = [&](auto j) -> cx<R> { return lds_at(j); };
        run_stages<R, RL, 0, L, TPL, true, false, SY>(u, tw, lds_at, zld, gst);
    } else if constexpr (IO == FK_IO_R2C_RR) {
        /* the real-to-real kinds that end in real outputs of an r2c of a line
           of N2 = 2L samples: R2HC, DHT, REDFT10 / RODFT10 (the line read in
           Makhoul's order) and REDFT00 / RODFT00 (the line read as its even /
           odd extension).  These passes have several 4- or 8-byte accesses
           and twiddles per element, so what bounds them is the latency and
           the number of their memory instructions: the choice of the kind is
           one branch around all loads and one around all stores, every
           element's address is a thread base plus a uniform offset, and the
           post-pass tables are read before the stages. */
        const R *inr = reinterpret_cast<const R *>(a.in) + bin;
        R *outr = reinterpret_cast<R *>(a.out) + bout;
        const cx<R> *wk = reinterpret_cast<const cx<R> *>(a.aux);
        const cx<R> *dt = reinterpret_cast<const cx<R> *>(a.rtw);
        const unsigned rm = a.rmode;
        const bool mak = rm == FK_RM_DCT2 || rm == FK_RM_DST2;
        const bool ext = rm == FK_RM_E00 || rm == FK_RM_O00;
        const long long is = a.is, os = a.os;
        constexpr long long N2 = 2LL * L;
        constexpr int R0 = RL::r[0], NB0 = L / R0;
        constexpr bool M0 = MirOk<RL, TPL>::first, SELF = MirOk<RL, TPL>::self;
        using BF = Bfly<NB0, TPL, M0>;
        constexpr int BPT = BF::BPT;
        /* elements j = b + r*NB0 of butterfly b: f(i, r, b) for those in range */
        auto each = [&](auto &&f) {
            sfor<0, BPT>([&](auto ic) {
                const int b = BF::template at<decltype(ic)::value>(u);
                if ((NB0 % TPL == 0) || b < NB0) sfor<0, R0>([&](auto rc) { f(ic, rc, b); });
            });
        };
        /* REDFT10 / RODFT10 read v_m = x_2m for m < L, x_{2(n-1-m)+1} above;
           the sine kind negates the odd samples (RODFT10_k(x) =
           REDFT10_{n-1-k}((-1)^j x_j)).  Samples 4j..4j+3 are elements j and
           L-1-j: v_2j, v_{n-1-2j}, v_{2j+1}, v_{n-2-2j}. */
        auto quads = [&](auto &v, auto &&quad) {
            sfor<0, BPT>([&](auto ic) {
                constexpr int i = decltype(ic)::value, im = SELF ? i : BF::image(i);
                const int b = BF::template at<i>(u);
                sfor<0, R0 / 2>([&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    R q[4];
                    quad(b, std::integral_constant<int, r * NB0>{}, q);
                    v[i][r] = mk(q[0], q[2]);
                    v[im][R0 - 1 - r] = mk(q[3], q[1]);
                });
            });
        };
        auto vld = [&](int m) -> R {
            const long long q = m < L ? 2LL * m : 2 * (N2 - 1 - m) + 1;
            return inr[q * is];
        };
        /* REDFT00 / RODFT00 read the even extension x_0..x_{n-1},
           x_{n-2}..x_1 (n = L+1) or the odd one 0, x_0..x_{n-1}, 0,
           -x_{n-1}..-x_0 (n = L-1) of the line */
        auto eld = [&](long long m) -> R {
            if (rm == FK_RM_E00) return inr[(m <= L ? m : N2 - m) * is];
            if (m == 0 || m == L) return (R)0;
            return m < L ? inr[(m - 1) * is] : -inr[(N2 - m - 1) * is];
        };
        auto first = whole([&](auto &v) {
            if (mak) {
                asm volatile("");
                if constexpr (M0 || SELF) {
                    if (fl & FK_REAL_QUAD) {
                        asm volatile("");
                        /* as pairs past L1 in FP32 (see FK_IO_R2C) */
                        struct alignas(16) Q { R x[16 / sizeof(R)]; };
                        auto fetch = [&](auto acc, auto *base) {
                            typedef typename std::decay<decltype(*base)>::type T;
                            constexpr int NT4 = 4 * sizeof(R) / sizeof(T), E = 4 / NT4;
                            quads(v, [&](int b, auto oc, R *q) {
                                const T *p = base + (b + decltype(oc)::value) * NT4;
                                sfor<0, NT4>([&](auto hc) {
                                    constexpr int h = decltype(hc)::value;
                                    const T x = ldg(acc, p + h);
                                    __builtin_memcpy(q + h * E, &x, sizeof(T));
                                });
                            });
                        };
                        if (nti) {
                            asm volatile("");
                            fetch(Acc<C_NT>{}, reinterpret_cast<const Q *>(inr));
                        } else if constexpr (sizeof(R) == 4) {
                            fetch(Acc<C_ONCE>{}, reinterpret_cast<const cx<R> *>(inr));
                        } else {
                            fetch(Acc<C_KEEP>{}, reinterpret_cast<const Q *>(inr));
                        }
                    } else {
                        quads(v, [&](int b, auto oc, R *q) {
                            const R *p = inr + 4 * b * is + (4LL * decltype(oc)::value) * is;
                            q[0] = p[0];
                            q[1] = p[is];
                            q[2] = p[2 * is];
                            q[3] = p[3 * is];
                        });
                    }
                } else {
                    each([&](auto ic, auto rc, int b) {
                        const int j = b + decltype(rc)::value * NB0;
                        v[decltype(ic)::value][decltype(rc)::value] = mk(vld(2 * j), vld(2 * j + 1));
                    });
                }
                if (rm == FK_RM_DST2) {
                    asm volatile("");
                    each([&](auto ic, auto rc, int b) {
                        constexpr int r = decltype(rc)::value;
                        cx<R> &x = v[decltype(ic)::value][r];
                        const int j = b + r * NB0;
                        if (R0 % 2 ? 2 * j >= L : 2 * r >= R0) x.x = -x.x;
                        if (R0 % 2 ? 2 * j + 1 >= L : 2 * r >= R0) x.y = -x.y;
                    });
                }
            } else if (ext) {
                asm volatile("");
                each([&](auto ic, auto rc, int b) {
                    constexpr int r = decltype(rc)::value;
                    cx<R> &x = v[decltype(ic)::value][r];
                    const int j = b + r * NB0;
                    if constexpr (R0 % 2 == 0 && r != 0 && 2 * r != R0) {
                        /* inside one half of the extension */
                        const long long sg = 2 * r < R0 ? is : -is;
                        const R *p = 2 * r < R0 ? inr + 2 * j * is - (rm == FK_RM_E00 ? 0 : is)
                                                : inr + (N2 - 2 * j) * is - (rm == FK_RM_E00 ? 0 : is);
                        x = mk(p[0], p[sg]);
                        if (2 * r > R0 && rm == FK_RM_O00) x = mk(-x.x, -x.y);
                    } else {
                        x = mk(eld(2 * j), eld(2 * j + 1));
                    }
                });
            } else if (fl & FK_REAL_UNIT) {
                /* past L1 where a line has 8 threads and more (see FK_IO_R2C;
                   R2HC of 64 samples, 4 threads, is a tenth faster through L1,
                   of 128 the same) */
                each([&](auto ic, auto rc, int b) {
                    constexpr int r = decltype(rc)::value;
                    v[decltype(ic)::value][r] =
                        ldg(Acc<(TPL >= 8 ? C_ONCE : C_KEEP)>{},
                            reinterpret_cast<const cx<R> *>(inr) + b + r * NB0);
                });
            } else {
                asm volatile("");
                each([&](auto ic, auto rc, int b) {
                    constexpr int r = decltype(rc)::value;
                    const R *p = inr + 2 * b * is + (2LL * r * NB0) * is;
                    v[decltype(ic)::value][r] = mk(p[0], p[is]);
                });
            }
        });
        auto lst = [&](auto k, cx<R> v) { lds_at(k) = v; };
        /* bins k = u + i*TPL <= L/2, with L-k: one table entry W_n^k each, for
           REDFT10 / RODFT10 also t_k and t_{L-k}, t_k = exp(-i pi k / 2n) */
        constexpr int HK = L / 2;
        constexpr int NK2 = (HK + 1 + TPL - 1) / TPL;
        constexpr bool PRE = NK2 * sizeof(R) <= 40 && NR <= 512;
        constexpr int GK = PRE ? NK2 : 4;
        struct W3 { cx<R> w, t, s; };
        W3 w[GK];
        auto tables = [&](auto gc) {
            sfor<0, GK>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                const int k = u + (decltype(gc)::value * GK + i) * TPL;
                w[i].w = wk[k <= HK ? k : HK];
            });
            if (mak) {
                asm volatile("");
                sfor<0, GK>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    const int k = u + (decltype(gc)::value * GK + i) * TPL;
                    w[i].t = dt[k <= HK ? k : HK];
                    w[i].s = dt[L - (k <= HK ? k : HK)];
                });
            }
        };
        if constexpr (PRE) tables(std::integral_constant<int, 0>{});
        run_stages<R, RL, 0, L, TPL, false, true, SY, M0>(u, tw, lds_at, first, lst);
        /* f(d, k, Z[k], Z[L-k], tables) with d = k - u a compile-time constant */
        auto bins = [&](auto gc, auto &&f) {
            sfor<0, GK>([&](auto ic) {
                constexpr int i = decltype(gc)::value * GK + decltype(ic)::value;
                const int k = u + i * TPL;
                if (act && i < NK2 && k <= HK)
                    f(std::integral_constant<int, i * TPL>{}, k, (cx<R>)lds_at(k),
                      (cx<R>)lds_at(k == 0 ? 0 : L - k), w[decltype(ic)::value]);
            });
        };
        /* X[k] = E + W O and X[L-k] = conj(E - W O), both rounding as the
           form of a bin on its own */
        auto XY = [&](cx<R> zk, cx<R> zc, cx<R> wv, cx<R> &X, cx<R> &Y) {
            const R er = (R)0.5 * (zk.x + zc.x), ei = (R)0.5 * (zk.y - zc.y);
            const R orr = (R)0.5 * (zk.y + zc.y), oi = (R)-0.5 * (zk.x - zc.x);
            X = mk(er + orr * wv.x - oi * wv.y, ei + orr * wv.y + oi * wv.x);
            Y = mk(er + orr * (-wv.x) - (-oi) * wv.y, (-ei) + orr * wv.y + (-oi) * (-wv.x));
        };
        /* outputs k, n-k, L-k, L+k (one lower for the sine kinds' mirror) */
        R *pk = outr + u * os, *pn = outr + (N2 - u) * os;
        R *pm = outr + (L - u) * os, *pp = outr + (L + u) * os;
        sfor<0, (NK2 + GK - 1) / GK>([&](auto gc) {
            if constexpr (!PRE) tables(gc);
            if (mak) {
                /* c_k = t_k X_k; REDFT10: y_k = 2 Re c_k, y_{n-k} = -2 Im c_k;
                   RODFT10: the same reversed */
                asm volatile("");
                const bool sn = rm == FK_RM_DST2;
                const long long st = sn ? -os : os;
                R *qk = sn ? outr + (N2 - 1 - u) * os : pk, *qn = sn ? pk - os : pn;
                R *qm = sn ? pp - os : pm, *qp = sn ? pm - os : pp;
                bins(gc, [&](auto dc, int k, cx<R> zk, cx<R> zc, const W3 &t) {
                    const long long d = (long long)decltype(dc)::value * st;
                    cx<R> X, Y;
                    XY(zk, zc, t.w, X, Y);
                    const cx<R> c = mul(X, t.t), e = mul(Y, t.s);
                    qk[d] = (R)2 * c.x;
                    if (k != 0) qn[-d] = (R)-2 * c.y;
                    if (2 * k != L) {
                        qm[-d] = (R)2 * e.x;
                        if (k != 0) qp[d] = (R)-2 * e.y;
                    }
                });
            } else if (ext) {
                /* DCT-I: Re X_k; DST-I: -Im X_k, one place lower */
                asm volatile("");
                bins(gc, [&](auto dc, int k, cx<R> zk, cx<R> zc, const W3 &t) {
                    const long long d = (long long)decltype(dc)::value * os;
                    cx<R> X, Y;
                    XY(zk, zc, t.w, X, Y);
                    if (rm == FK_RM_E00) {
                        pk[d] = X.x;
                        if (2 * k != L) pm[-d] = Y.x;
                    } else if (k != 0) {
                        pk[d - os] = -X.y;
                        if (2 * k != L) pm[-d - os] = -Y.y;
                    }
                });
            } else {
                /* R2HC: r_k, i_k; DHT: Re - Im, Re + Im, at k and n-k */
                bins(gc, [&](auto dc, int k, cx<R> zk, cx<R> zc, const W3 &t) {
                    const long long d = (long long)decltype(dc)::value * os;
                    cx<R> X, Y;
                    XY(zk, zc, t.w, X, Y);
                    if (rm == FK_RM_DHT) {
                        X = mk(X.x - X.y, X.x + X.y);
                        Y = mk(Y.x - Y.y, Y.x + Y.y);
                    }
                    pk[d] = X.x;
                    if (k != 0) pn[-d] = X.y;
                    if (2 * k != L) {
                        pm[-d] = Y.x;
                        if (k != 0) pp[d] = Y.y;
                    }
                });
            }
        });
    } else if constexpr (IO == FK_IO_C2R_RR) {
        /* the real-to-real kinds that begin with real inputs of a c2r: HC2R
           (bins r_k, i_k from the halfcomplex line), REDFT01 / RODFT01 (bins
           V_k = exp(+i pi k / 2n)(x_k - i x_{n-k}), the sine kind on the
           reversed line; outputs y_2i = v_i, y_2i+1 = v_{n-1-i}, the sine
           kind's odd ones negated).  Bounded as the kinds above. */
        const R *inr = reinterpret_cast<const R *>(a.in) + bin;
        R *outr = reinterpret_cast<R *>(a.out) + bout;
        const cx<R> *wk = reinterpret_cast<const cx<R> *>(a.aux);
        const cx<R> *dt = reinterpret_cast<const cx<R> *>(a.rtw);
        const bool hc = a.rmode == FK_RM_HC2R, sn = a.rmode == FK_RM_DST3;
        const long long is = a.is, os = a.os;
        constexpr long long N2 = 2LL * L;
        constexpr int HK = L / 2;
        constexpr int NK2 = (HK + 1 + TPL - 1) / TPL;
        constexpr int GK = sizeof(R) == 4 ? 9 : 4;
        struct W3 { cx<R> w, t, s; };
        /* samples k, n-k, L-k, L+k of the line (reversed for RODFT01) */
        const long long st = sn ? -is : is, o = sn ? N2 - 1 : 0;
        const R *pk = inr + o * is + u * st, *pn = inr + o * is + (N2 - u) * st;
        const R *pm = inr + o * is + (L - u) * st, *pp = inr + o * is + (L + u) * st;
        sfor<0, (NK2 + GK - 1) / GK>([&](auto gc) {
            constexpr int g = decltype(gc)::value;
            constexpr int cnt = (NK2 - g * GK) < GK ? (NK2 - g * GK) : GK;
            R xk[cnt], xn[cnt], xm[cnt], xp[cnt];
            W3 w[cnt];
            sfor<0, cnt>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                const int k = u + (g * GK + i) * TPL;
                const long long d = (long long)((g * GK + i) * TPL) * st;
                if (k <= HK) {
                    xk[i] = pk[d];
                    xn[i] = k == 0 ? (R)0 : pn[-d];
                    xm[i] = pm[-d];
                    xp[i] = pp[d];
                }
            });
            sfor<0, cnt>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                const int k = u + (g * GK + i) * TPL;
                w[i].w = wk[k <= HK ? k : HK];
            });
            cx<R> X[cnt], Y[cnt];
            if (hc) {
                /* X[k] = (x_k, x_{n-k}), X[L-k] = (x_{L-k}, x_{L+k}),
                   Im X[0] = Im X[L] = 0 */
                sfor<0, cnt>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    const int k = u + (g * GK + i) * TPL;
                    X[i] = mk(xk[i], xn[i]);
                    Y[i] = mk(xm[i], k == 0 ? (R)0 : xp[i]);
                });
            } else {
                /* V_k = conj(t_k) (x_k - i x_{n-k}), t_k = exp(-i pi k / 2n) */
                asm volatile("");
                sfor<0, cnt>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    const int k = u + (g * GK + i) * TPL;
                    w[i].t = dt[k <= HK ? k : HK];
                    w[i].s = dt[L - (k <= HK ? k : HK)];
                });
                sfor<0, cnt>([&](auto ic) {
                    constexpr int i = decltype(ic)::value;
                    const int k = u + (g * GK + i) * TPL;
                    const cx<R> t = w[i].t, t2 = w[i].s;
                    X[i] = mk(t.x * xk[i] - t.y * xn[i], -(t.x * xn[i] + t.y * xk[i]));
                    Y[i] = mk(t2.x * xm[i] - t2.y * xp[i], -(t2.x * xp[i] + t2.y * xm[i]));
                    /* Im V_0 = Im V_L = 0 */
                    if (k == 0) X[i].y = Y[i].y = 0;
                });
            }
            /* as in FK_IO_C2R, swapped: e = X[k] + conj X[L-k], o = (X[k] -
               conj X[L-k]) conj(W_n^k), Z[k] = e + i o, Z[L-k] = conj e + i conj o */
            sfor<0, cnt>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                const int k = u + (g * GK + i) * TPL;
                if (k <= HK) {
                    const cx<R> e = mk(X[i].x + Y[i].x, X[i].y - Y[i].y);
                    const cx<R> d = mk(X[i].x - Y[i].x, X[i].y + Y[i].y), t = w[i].w;
                    const cx<R> o2 = mk(d.x * t.x + d.y * t.y, d.y * t.x - d.x * t.y);
                    lds_at(k) = mk(e.y + o2.x, e.x - o2.y);
                    if (k != 0 && 2 * k != L) lds_at(L - k) = mk(o2.x - e.y, e.x + o2.y);
                }
            });
        });
        SY::sync();
        constexpr int RN = RL::r[RL::n - 1], NBN = L / RN;
        constexpr bool ML = MirOk<RL, TPL>::last, SELF = MirOk<RL, TPL>::self;
        using BF = Bfly<NBN, TPL, ML>;
        constexpr int BPT = BF::BPT;
        /* v = swap(z_k): (v_2k+1, v_2k) */
        auto last = whole([&](auto &v) {
            auto each = [&](auto &&f) {
                sfor<0, BPT>([&](auto ic) {
                    const int b = BF::template at<decltype(ic)::value>(u);
                    if (act && ((NBN % TPL == 0) || b < NBN))
                        sfor<0, RN>([&](auto rc) {
                            constexpr int r = decltype(rc)::value;
                            f(b, std::integral_constant<int, r * NBN>{}, v[decltype(ic)::value][r]);
                        });
                });
            };
            if (!hc) {
                asm volatile("");
                if constexpr (ML || SELF) {
                    /* elements k and L-1-k are outputs 4k..4k+3 */
                    auto quads = [&](auto &&quad) {
                        if (act)
                            sfor<0, BPT>([&](auto ic) {
                                constexpr int i = decltype(ic)::value, im = SELF ? i : BF::image(i);
                                const int b = BF::template at<i>(u);
                                sfor<0, RN / 2>([&](auto rc) {
                                    constexpr int r = decltype(rc)::value;
                                    const cx<R> x = v[i][r], y = v[im][RN - 1 - r];
                                    const R y1 = sn ? -y.x : y.x, y3 = sn ? -y.y : y.y;
                                    const R q[4] = {x.y, y1, x.x, y3};
                                    quad(b, std::integral_constant<int, r * NBN>{}, q);
                                });
                            });
                    };
                    if (fl & FK_REAL_QUAD) {
                        asm volatile("");
                        struct alignas(16) Q { R x[16 / sizeof(R)]; };
                        constexpr int NQ = sizeof(R) / 4;
                        Q *q4 = reinterpret_cast<Q *>(outr);
                        quads([&](int b, auto oc, const R *q) {
                            Q *p = q4 + (b + decltype(oc)::value) * NQ;
                            sfor<0, NQ>([&](auto hc_) {
                                constexpr int hh = decltype(hc_)::value;
                                Q x;
                                sfor<0, 4 / NQ>([&](auto ec) {
                                    constexpr int e = decltype(ec)::value;
                                    x.x[e] = q[hh * (4 / NQ) + e];
                                });
                                p[hh] = x;
                            });
                        });
                    } else {
                        quads([&](int b, auto oc, const R *q) {
                            R *p = outr + 4 * b * os + (4LL * decltype(oc)::value) * os;
                            p[0] = q[0];
                            p[os] = q[1];
                            p[2 * os] = q[2];
                            p[3 * os] = q[3];
                        });
                    }
                } else {
                    each([&](int b, auto oc, cx<R> x) {
                        const long long m0 = 2LL * (b + decltype(oc)::value), m1 = m0 + 1;
                        const long long d0 = m0 < L ? 2 * m0 : 2 * (N2 - 1 - m0) + 1;
                        const long long d1 = m1 < L ? 2 * m1 : 2 * (N2 - 1 - m1) + 1;
                        outr[d0 * os] = (sn && (d0 & 1)) ? -x.y : x.y;
                        outr[d1 * os] = (sn && (d1 & 1)) ? -x.x : x.x;
                    });
                }
            } else if (fl & FK_REAL_UNIT) {
                each([&](int b, auto oc, cx<R> x) {
                    reinterpret_cast<cx<R> *>(outr)[b + decltype(oc)::value] = mk(x.y, x.x);
                });
            } else {
                asm volatile("");
                each([&](int b, auto oc, cx<R> x) {
                    R *p = outr + 2 * b * os + (2LL * decltype(oc)::value) * os;
                    p[0] = x.y;
                    p[os] = x.x;
                });
            }
        });
        auto zld = [&](auto j) -> cx<R> { return lds_at(j); };
        run_stages<R, RL, 0, L, TPL, true, false, SY, false, ML>(u, tw, lds_at, zld, last);
    } else if constexpr (IO == FK_IO_BLUE) {
        /* Bluestein (dft/bluestein.c:82-128 conventions): a_j = x_j c_j,
           c_j = exp(-i pi j^2/n); conv = IDFT_L(DFT_L(a) * B),
           B = DFT_L(conj c)/L; y_k = c_k conv_k, k < n. */
        const cx<R> *in = reinterpret_cast<const cx<R> *>(a.in) + bin;
        cx<R> *out = reinterpret_cast<cx<R> *>(a.out);
        const cx<R> *chirp = reinterpret_cast<const cx<R> *>(a.aux);
        const cx<R> *Bt = reinterpret_cast<const cx<R> *>(a.aux2);
        const int n = (int)a.nvalid;
        auto gld = [&](int j) -> cx<R> {
            if (!act || j >= n) return mk((R)0, (R)0);
            cx<R> v = in[j * a.is];
            if (swi) v = swp(v);
            return mul(v, chirp[j]);
        };
        auto lst = [&](auto k, cx<R> v) { lds_at(k) = v; };
        run_stages<R, RL, 0, L, TPL, false, true, SY>(u, tw, lds_at, gld, lst);
        auto mid = [&](int j) -> cx<R> { return swp(mul(lds_at(j), Bt[j])); };
        auto gst = [&](int k, cx<R> v) {
            if (k < n && act) {
                const cx<R> y = mul(swp(v), chirp[k]);
                out[bout + k * a.os] = swo ? swp(y) : y;
            }
        };
        run_stages<R, RL, 0, L, TPL, true, false, SY>(u, tw, lds_at, mid, gst);
    }
}

template <typename R, int NL, int MODE, int IO, int PAD, class RL, int TPL>
__global__ void __launch_bounds__(TPL * NL)
stockham(fk_args a)
{
    extern __shared__ unsigned char smem_raw[];
    /* row mapping with whole lines inside one wave: wave-level exchange */
    constexpr bool wave_lines = MODE == FK_ROW && TPL <= 64 && 64 % TPL == 0;
    using SY = typename std::conditional<wave_lines, SyncWave, SyncAll>::type;
    stockham_body<R, NL, MODE, IO, PAD, RL, TPL, TPL * NL, SY>(a, remap_tile(a.xcd_remap),
                                                               smem_raw);
}

/*
 * Row-mapped plain pass with one stage-0 butterfly per thread (L / R0 =
 * TPL) whose workgroups each run several tiles: the grid holds the
 * workgroups the device keeps resident, a workgroup steps through tiles
 * blockIdx.x + k*gridDim.x, and the next tile's stage-0 inputs are loaded
 * into registers while the current tile runs its stages, so HBM reads
 * overlap the LDS stages that otherwise follow each tile's loads.  For
 * long lines (one or a few per workgroup) the whole batch is only a couple
 * of workgroup rounds, which stockham<> runs with load, compute and store
 * phases in lock-step.  Same arithmetic as stockham<>: identical output.
 */
template <typename R, int NL, int PAD, class RL, int TPL>
__global__ void __launch_bounds__(TPL * NL, 4)
stockham_pipe(fk_args a)
{
    constexpr int L = RL::L(), R0 = RL::r[0], NB0 = L / R0;
    static_assert(NB0 == TPL, "one stage-0 butterfly per thread");
    using G = Geo<R, L, TPL, NL, FK_ROW, PAD>;
    constexpr bool wave_lines = TPL <= 64 && 64 % TPL == 0;
    using SY = typename std::conditional<wave_lines, SyncWave, SyncAll>::type;
    extern __shared__ unsigned char smem_raw[];
    cx<R> *lds = reinterpret_cast<cx<R> *>(smem_raw);
    const int tid = threadIdx.x, u = tid % TPL;
    const int lt = TPL % 64 == 0 ? __builtin_amdgcn_readfirstlane(tid / TPL) : tid / TPL;
    const long long ntiles = (a.nlines + NL - 1) / NL, step = gridDim.x;
    const unsigned fl = a.flags;
    const bool swi = fl & FK_SWAP_IN, swo = fl & FK_SWAP_OUT;
    const long long is = a.is, os = a.os;
    const cx<R> *tw = reinterpret_cast<const cx<R> *>(a.tw);
    const cx<R> *in = reinterpret_cast<const cx<R> *>(a.in);
    cx<R> *out = reinterpret_cast<cx<R> *>(a.out);
    /* line of tile t for this thread: input and output offsets, computed
       once per tile when its inputs are fetched; lanes past the last line
       use line 0 (in bounds) and store nothing */
    auto line_of = [&](long long t, long long &bin, long long &bout) -> bool {
        const long long line = t * NL + lt;
        const bool act = line < a.nlines;
        line_off(a, line_ix(a, act ? line : 0), bin, bout);
        return act;
    };
    long long t = blockIdx.x;
    if (t >= ntiles) return;
    cx<R> cur[R0], nxt[R0];
    /* stage-0 inputs of the thread's butterfly */
    auto fetch = [&](long long bin, cx<R> *v) {
        const cx<R> *p = in + bin + u * is;
        with_acc(sizeof(R) == 8 && (fl & FK_NT_IN), [&](auto acc) {
            sfor<0, R0>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                v[r] = ldg(acc, p + (long long)(r * NB0) * is);
            });
        });
    };
    long long bin, bout;
    bool act = line_of(t, bin, bout);
    fetch(bin, cur);
    auto lds_at = [&](auto j) -> cx<R> & { return lds[G::idx(lt, j)]; };
    for (;;) {
        const long long tn = t + step;
        const bool more = tn < ntiles;
        long long bin_n = 0, bout_n = 0;
        bool act_n = false;
        if (more) {
            act_n = line_of(tn, bin_n, bout_n);
            fetch(bin_n, nxt);
        }
        cx<R> *outu = out + bout + u * os;
        auto first = [&](auto j) -> cx<R> {
            constexpr int r = AtOff<typename std::decay<decltype(j)>::type>::v / NB0;
            return cur[r];
        };
        auto gst = hoisted([&](auto &&store) {
            with_acc(sizeof(R) == 8 && (fl & FK_NT_OUT), [&](auto acc) {
                store([&](int k, cx<R> v) {
                    if (NL == 1 || act) stg(acc, outu + (long long)(k - u) * os, v);
                });
            });
        });
        /* no four-step twiddle here: the planner runs passes that need it
           with stockham<> */
        run_stages<R, RL, 0, L, TPL, false, false, SY>(u, tw, lds_at, first, gst, SwapOp{swi},
                                                       SwapOp{swo});
        if (!more) break;
        sfor<0, R0>([&](auto rc) {
            constexpr int r = decltype(rc)::value;
            cur[r] = nxt[r];
        });
        t = tn;
        bout = bout_n;
        act = act_n;
        /* the next tile's stage-0 LDS writes follow every read of this one */
        __syncthreads();
    }
}

/*
 * Row-mapped plain pass whose LDS exchange moves the real parts, then the
 * imaginary parts, through one array of reals: half the LDS per line of
 * stockham<> (more workgroups resident per CU to hide HBM latency) for
 * four workgroup barriers per exchange instead of two.  Stage s computes in
 * registers, writes its outputs' real parts, every thread reads the real
 * parts of its next-stage inputs, then the same for the imaginary parts.
 */
template <class RL, int S, int L, int TPL>
struct XsGeo {
    static constexpr int Rs = RL::r[S];
    static constexpr int Ns = RL::ns(S);
    static constexpr int NB = L / Rs;
    static constexpr int BPT = (NB + TPL - 1) / TPL;
};

template <typename R, class RL, int S, int L, int TPL, class PosF, class LastF, class FinF>
__device__ __forceinline__ void run_xs(int u, const cx<R> *__restrict__ tw, R *buf, PosF &&idx,
                                       cx<R> (&v)[XsGeo<RL, S, L, TPL>::BPT][XsGeo<RL, S, L, TPL>::Rs],
                                       LastF &&last, const FinF &fin)
{
    using X = XsGeo<RL, S, L, TPL>;
    constexpr int Rs = X::Rs, Ns = X::Ns, NB = X::NB, BPT = X::BPT;
    sfor<0, BPT>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const int b = u + i * TPL;
        if ((NB % TPL == 0) || b < NB) {
            if constexpr (S > 0) {
                const int k = b % Ns;
                const cx<R> *w = tw + RL::twoff(S) + k * (Rs - 1);
                sfor<1, Rs>([&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    v[i][r] = mul(v[i][r], w[r - 1]);
                });
            }
            Dft<R, Rs, 1>::run(v[i]);
            if constexpr (S == RL::n - 1) fin.template run<Rs, i>(b, v[i]);
        }
    });
    auto each_out = [&](auto &&f) {
        sfor<0, BPT>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const int b = u + i * TPL;
            if ((NB % TPL == 0) || b < NB) {
                const int k = b % Ns, base = (b - k) * Rs + k;
                sfor<0, Rs>([&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    f(base + r * Ns, v[i][r]);
                });
            }
        });
    };
    if constexpr (S == RL::n - 1) {
        each_out([&](int k, cx<R> x) { last(k, x); });
    } else {
        using Y = XsGeo<RL, S + 1, L, TPL>;
        cx<R> w[Y::BPT][Y::Rs];
        auto each_in = [&](auto &&f) {
            sfor<0, Y::BPT>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                const int b = u + i * TPL;
                if ((Y::NB % TPL == 0) || b < Y::NB) {
                    sfor<0, Y::Rs>([&](auto rc) {
                        constexpr int r = decltype(rc)::value;
                        f(b + r * Y::NB, w[i][r]);
                    });
                }
            });
        };
        each_out([&](int k, cx<R> x) { buf[idx(k)] = x.x; });
        __syncthreads();
        each_in([&](int j, cx<R> &x) { x.x = buf[idx(j)]; });
        __syncthreads();
        each_out([&](int k, cx<R> x) { buf[idx(k)] = x.y; });
        __syncthreads();
        each_in([&](int j, cx<R> &x) { x.y = buf[idx(j)]; });
        __syncthreads();
        run_xs<R, RL, S + 1, L, TPL>(u, tw, buf, idx, w, last, fin);
    }
}

template <typename R, int NL, int MODE, int PAD, class RL, int TPL>
__global__ void __launch_bounds__(TPL * NL)
stockham_xs(fk_args a)
{
    extern __shared__ unsigned char smem_raw[];
    constexpr int L = RL::L();
    constexpr int LP = L + L / PAD + 2;
    const long long tile = remap_tile(a.xcd_remap);
    /* row mapping: a line's threads are consecutive, its reals one padded
       LDS row; column mapping: consecutive threads are consecutive lines
       (unit-stride batch), LDS laid out [element][line] */
    const int tid = threadIdx.x;
    const int lt = MODE == FK_ROW ? tid / TPL : tid % NL;
    const int u = MODE == FK_ROW ? tid % TPL : tid / NL;
    const long long line = tile * NL + lt;
    const bool act = line < a.nlines;
    const LineIx lx = line_ix(a, act ? line : 0);
    long long bin, bout;
    line_off(a, lx, bin, bout);
    const cx<R> *tw = reinterpret_cast<const cx<R> *>(a.tw);
    const cx<R> *in = reinterpret_cast<const cx<R> *>(a.in) + bin;
    cx<R> *out = reinterpret_cast<cx<R> *>(a.out);
    const unsigned fl = a.flags;
    const bool swi = fl & FK_SWAP_IN;
    R *buf = reinterpret_cast<R *>(smem_raw) + (MODE == FK_ROW ? lt * LP : lt);
    auto idx = [](int j) { return MODE == FK_ROW ? j + j / PAD : j * NL; };
    const PlainOut<R, RL, TPL> fin(a, fl, lx.i0, u);
    auto gst = [&](int k, cx<R> v) {
        if (act) out[bout + k * a.os] = v;
    };
    using X0 = XsGeo<RL, 0, L, TPL>;
    cx<R> v[X0::BPT][X0::Rs];
    sfor<0, X0::BPT>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const int b = u + i * TPL;
        if ((X0::NB % TPL == 0) || b < X0::NB) {
            sfor<0, X0::Rs>([&](auto rc) {
                constexpr int r = decltype(rc)::value;
                cx<R> x = act ? in[(long long)(b + r * X0::NB) * a.is] : mk((R)0, (R)0);
                v[i][r] = swi ? swp(x) : x;
            });
        }
    });
    run_xs<R, RL, 0, L, TPL>(u, tw, buf, idx, v, gst, fin);
}

template <typename R, int NL, int MODE, int PAD, class RL, int TPL>
constexpr unsigned stockham_xs_lds()
{
    return (unsigned)(NL * (MODE == FK_ROW ? RL::L() + RL::L() / PAD + 2 : RL::L()) * sizeof(R));
}

template <typename R, int NL, int MODE, int IO, int PAD, class RL, int TPL, int NT = TPL * NL>
constexpr unsigned stockham_lds()
{
    using G = Geo<R, RL::L(), TPL, NL, MODE, PAD>;
    return G::lds_elems() * sizeof(cx<R>) + ((NL + 1) & ~1) * sizeof(long long) +
           (NT > TPL * NL ? 64 * sizeof(cx<R>) : 0);
}

} // namespace fk
#endif
