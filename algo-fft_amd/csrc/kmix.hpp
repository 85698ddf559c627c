// Runtime-size Stockham kernels for 2/3/5/7-smooth lengths with composite
// radices up to 20 (the mixed-radix path; the reference's mixedradix.go:45-358
// does the same recursion depth-first on the CPU and sends 7-smooth sizes to
// Bluestein instead).
//
// A block holds G transforms of N points in one LDS buffer, TPT threads each
// (the host's mix_config picks the radices, TPT and G).  The first pass reads
// global memory straight into registers and the last one writes its outputs
// straight to global memory, so P passes cost P - 1 trips through LDS; the
// passes between work in place (read all of a thread's butterflies, barrier,
// write).
//
// What bounds it: HBM for most lengths up to 10000 points, then the number
// of waves that one or two blocks a CU leave in flight.  Against one radix
// of {2, 3, 4, 5, 7, 8, 16} per pass the composite radices halve the passes
// (3000 = 20 x 10 x 15 instead of 3 x 5 x 5 x 5 x 8).  512 MiB complex64
// batches, before -> now: rows 1000 0.248 -> 0.19 ms, 3000 0.342 -> 0.20,
// 6000 0.365 -> 0.22, 8000 0.334 -> 0.19, 12000 0.475 -> 0.29 (a copy kernel
// of that pattern: 0.17); strided axes of 1000 points 0.34 -> 0.27.
#pragma once
#include "kernels.hpp"

namespace afft {

constexpr int MIX_MAXPASS = 8;
constexpr int MIX_RMAX = 20;   // largest radix

struct MixPass {
    int rad, ns, nr;      // radix, Ns = product of the earlier radices, N / rad
    unsigned nsm;         // mod_magic(ns)
    int twoff;            // first entry of the pass's twiddles
};

struct MixArgs {
    KArgs k;
    int n, npass;
    MixPass p[MIX_MAXPASS];
    int tpt;              // threads per transform
    int g;                // transforms per block (a power of two for VAR_4B)
    unsigned divm;        // mod_magic(tpt) for row layouts, mod_magic(g) for columns
    int pitch;            // LDS row pitch (row layouts)
};

// Butterflies of radix R that a thread may hold in one pass: 12 to 21 points,
// at least 16 for every radix from 2 to 10, so a schedule of at most N/16
// threads a transform always exists.
__host__ __device__ constexpr int mix_mb(int R) {
    return R >= 12 ? 1 : R >= 8 ? 2 : R >= 6 ? 3 : R == 5 ? 4 : R == 4 ? 5 : R == 3 ? 6 : 8;
}

// Largest blocks: complex64 needs 88-96 VGPRs (5 waves per SIMD), complex128
// 168-177 (2-3 waves).
template <typename T>
struct MixCfg {
    static constexpr int THREADS = sizeof(T) == 4 ? 1024 : 512;
    static constexpr int WAVES = sizeof(T) == 4 ? 4 : 2;   // per SIMD, at least
};

// Twiddle entries loaded per butterfly: every power for radices up to 8, else
// w^1, w^2, w^3 and w^4, w^8, w^12, w^16, whose products give the others (one
// product each).  Entry i * Ns + k of the pass's table is the i-th of them for
// butterfly k; tw is a const cx<T>* or a gptr<cx<T>>.  A radix-10 butterfly loads 5 values instead of 9: with every
// power loaded complex64 rows of 960 points took 0.233 ms instead of 0.203,
// complex128 rows of 1500 0.236 instead of 0.209.  Issuing the loads before
// the barrier in front of the pass lost 2-8 % (registers).  Fewer loads (w^1,
// w^2, w^4, ... and up to three products) were no faster and cost 1-3 % in
// error.
__host__ __device__ constexpr int mix_ntw(int R) { return R <= 8 ? R - 1 : 3 + (R - 1) / 4; }
__host__ __device__ constexpr int mix_twpow(int R, int i) { return R <= 8 || i < 3 ? i + 1 : 4 * (i - 2); }

template <int R, int DIR, typename T, class W>
__device__ __forceinline__ void mix_twiddle(W tw, int NS, int k, cx<T>* v) {
    constexpr int NW = mix_ntw(R);
    cx<T> w[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) w[i] = (tw + i * NS)[(unsigned)k];
#pragma unroll
    for (int r = 1; r < R; ++r) {
        if constexpr (R <= 8) {
            v[r] = twmul<DIR>(v[r], w[r - 1]);
        } else {
            const int q = r / 4, m = r % 4;
            const cx<T> ww = q == 0 ? w[m - 1] : m == 0 ? w[q + 2] : cmul(w[q + 2], w[m - 1]);
            v[r] = twmul<DIR>(v[r], ww);
        }
    }
}

// j / d and j mod d from m = mod_magic(d) (see fast_mod).
__device__ __forceinline__ int fast_divmod(int j, int d, unsigned m, int* rem) {
    unsigned q = __umulhi((unsigned)j, m);
    int r = j - (int)(q * (unsigned)d);
    if (r >= d) { r -= d; ++q; }
    *rem = r;
    return (int)q;
}

// One radix-R pass: thread t of TPT takes butterflies j = t, t + TPT, ... <
// N/R; load(v, j, NR) reads points j + r*NR, store(v, base, NS) takes points
// base + r*NS.  FIRST: no twiddles (Ns = 1).  HOLD: all of the thread's
// butterflies are read before bar() and stored after it; otherwise one after
// the other.  Every thread of the block calls this.
template <int R, int DIR, bool FIRST, bool HOLD, typename T, class W, class Load, class Store, class Bar>
__device__ __forceinline__ void mix_pass(bool act, int t, int TPT, const MixPass& ps, W tw, Load load, Store store,
                                         Bar bar) {
    constexpr int MB = mix_mb(R);
    const int NR = ps.nr, NS = ps.ns;
    if constexpr (HOLD || MB == 1) {
        cx<T> v[MB][R];
        int k[MB];
#pragma unroll
        for (int b = 0; b < MB; ++b) {
            const int j = t + b * TPT;
            k[b] = 0;
            if (act && j < NR) {
                load(v[b], j, NR);
                if constexpr (!FIRST) {
                    k[b] = fast_mod(j, NS, ps.nsm);
                    mix_twiddle<R, DIR>(tw, NS, k[b], v[b]);
                }
                dft<R, DIR, 1>(v[b]);
            }
        }
        bar();
#pragma unroll
        for (int b = 0; b < MB; ++b) {
            const int j = t + b * TPT;
            if (act && j < NR) store(v[b], FIRST ? j * R : (j - k[b]) * R + k[b], NS);
        }
    } else if (act) {
        for (int j = t; j < NR; j += TPT) {
            cx<T> v[R];
            load(v, j, NR);
            int k = 0;
            if constexpr (!FIRST) {
                k = fast_mod(j, NS, ps.nsm);
                mix_twiddle<R, DIR>(tw, NS, k, v);
            }
            dft<R, DIR, 1>(v);
            store(v, FIRST ? j * R : (j - k) * R + k, NS);
        }
    }
}

template <int DIR, bool FIRST, bool HOLD, typename T, class W, class Load, class Store, class Bar>
__device__ __forceinline__ void mix_pass_any(bool act, int t, int TPT, const MixPass& ps, W tw, Load load,
                                             Store store, Bar bar) {
#define AFFT_MIX_CASE(RR) \
    case RR: mix_pass<RR, DIR, FIRST, HOLD, T>(act, t, TPT, ps, tw, load, store, bar); break;
    switch (ps.rad) {
        AFFT_MIX_CASE(2)
        AFFT_MIX_CASE(3)
        AFFT_MIX_CASE(4)
        AFFT_MIX_CASE(5)
        AFFT_MIX_CASE(6)
        AFFT_MIX_CASE(7)
        AFFT_MIX_CASE(8)
        AFFT_MIX_CASE(9)
        AFFT_MIX_CASE(10)
        AFFT_MIX_CASE(12)
        AFFT_MIX_CASE(14)
        AFFT_MIX_CASE(15)
        AFFT_MIX_CASE(16)
        AFFT_MIX_CASE(18)
        AFFT_MIX_CASE(20)
    default: break;
    }
#undef AFFT_MIX_CASE
}

// All passes: the first reads through first(v, j, NR) and the last hands its
// outputs to last(v, base, NS) with the lane mapping (actl, tl, rowl) of that
// side.  LDS point n of this thread's transform sits at row[n * pn] (rowl for
// the last pass's reads).  LHOLD holds all of a thread's last-pass butterflies
// in flight before it stores the first.
template <typename T, int DIR, bool LHOLD, class First, class Last>
__device__ __forceinline__ void mix_transform(const MixArgs& g, const cx<T>* __restrict__ tw, bool act, int t,
                                              cx<T>* row, bool actl, int tl, cx<T>* rowl, int pn, First first,
                                              Last last) {
    const int TPT = g.tpt, np = g.npass - 1;
    auto load_s = [&](auto& v, int j, int NR) __attribute__((always_inline)) {
        constexpr int R = sizeof(v) / sizeof(v[0]);
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = row[(j + r * NR) * pn];
    };
    auto load_l = [&](auto& v, int j, int NR) __attribute__((always_inline)) {
        constexpr int R = sizeof(v) / sizeof(v[0]);
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = rowl[(j + r * NR) * pn];
    };
    auto store_s = [&](auto& v, int base, int NS) __attribute__((always_inline)) {
        constexpr int R = sizeof(v) / sizeof(v[0]);
#pragma unroll
        for (int r = 0; r < R; ++r) row[(base + r * NS) * pn] = v[r];
    };
    auto sync = [] { __syncthreads(); };
    auto none = [] {};
    if (np == 0) {
        mix_pass_any<DIR, true, false, T>(act, t, TPT, g.p[0], tw, first, last, none);
        return;
    }
    mix_pass_any<DIR, true, true, T>(act, t, TPT, g.p[0], tw, first, store_s, none);
    __syncthreads();
    for (int p = 1; p < np; ++p) {
        mix_pass_any<DIR, false, true, T>(act, t, TPT, g.p[p], tw + g.p[p].twoff, load_s, store_s, sync);
        __syncthreads();
    }
    mix_pass_any<DIR, false, LHOLD, T>(actl, tl, TPT, g.p[np], tw + g.p[np].twoff, load_l, last, none);
}

// VAR_ROW / VAR_COL / VAR_4A / VAR_4B as in kernels.hpp.  Row layouts keep
// transform c at sm[c * pitch ..] with lanes along its points, column layouts
// interleave the G columns with lanes along them.  VAR_4B reads rows with
// lanes along n and runs its last pass with lanes along c (an odd pitch keeps
// those reads free of bank conflicts), so its transposing store needs no
// extra trip through LDS.
template <typename T, int VAR, int DIR>
__global__ void __launch_bounds__(MixCfg<T>::THREADS, MixCfg<T>::WAVES) k_mix(MixArgs g) {
    extern __shared__ unsigned char smraw[];
    cx<T>* sm = (cx<T>*)smraw;
    const KArgs a = g.k;
    constexpr bool COLL = VAR == VAR_COL || VAR == VAR_4A;
    const int G = g.g, TPT = g.tpt, tid = threadIdx.x, P = g.pitch;
    int c, t;
    if constexpr (COLL) t = fast_divmod(tid, G, g.divm, &c);
    else c = fast_divmod(tid, TPT, g.divm, &t);
    // Neighbouring column groups share cache lines unless they start and end
    // on line boundaries: blocks in XCD order keep them in one L2.  Columns
    // of 8 complex64 (half lines), rows of 512: 1200 points 0.339 -> 0.275 ms, 2000 0.344 ->
    // 0.296; 16 columns, rows of 961: 500 points 0.354 -> 0.266; transposing
    // stores (VAR_4B), rows of 500: 400 points 0.318 -> 0.251.
    unsigned bx = blockIdx.x, by = blockIdx.y;
    if constexpr (VAR != VAR_ROW) xcd_block(&bx, &by);
    const long long c0 = (long long)bx * G;
    const bool act = tid < G * TPT && c0 + c < a.count;
    const cx<T>* __restrict__ in = (const cx<T>*)a.in + (long long)by * a.in_bd;
    cx<T>* __restrict__ out = (cx<T>*)a.out + (long long)by * a.out_bd;
    const cx<T>* __restrict__ tw = (const cx<T>*)a.tw;
    const cx<T>* src = COLL ? in + (c0 + c) : in + (c0 + c) * a.in_cd;
    const long long ind = COLL ? a.in_nd : 1;
    const int nt = a.nt;
    auto load_g = [&](auto& v, int j, int NR) __attribute__((always_inline)) {
        constexpr int R = sizeof(v) / sizeof(v[0]);
        const cx<T>* q = src + (long long)j * ind;
        const long long st = (long long)NR * ind;
        if (nt & NT_LOAD) {
#pragma unroll
            for (int r = 0; r < R; ++r, q += st) v[r] = ld_nt(q);
        } else {
#pragma unroll
            for (int r = 0; r < R; ++r, q += st) v[r] = *q;
        }
    };
    int cl = c, tl = t;
    if constexpr (VAR == VAR_4B) {
        cl = tid & (G - 1);
        tl = tid >> (__ffs(G) - 1);
    }
    const bool actl = tid < G * TPT && c0 + cl < a.count;
    cx<T>* dst = VAR == VAR_ROW ? out + (c0 + cl) * a.out_cd : out + (c0 + cl);
    const long long ond = VAR == VAR_ROW ? 1 : a.out_nd;
    auto store_g = [&](auto& v, int base, int NS) __attribute__((always_inline)) {
        constexpr int R = sizeof(v) / sizeof(v[0]);
        if constexpr (VAR == VAR_4A) {
            // W_L^{k*col} for k = base + r*Ns from a table value and the step
            // W_L^{Ns*col} (lanes differ in col, so the table gathers hit
            // scattered lines).  complex64 steps in double from tables in
            // double and rounds each factor once: a value and a step a
            // butterfly.  Float tables with a value every fourth r took
            // 1-2.5 % longer and put the products' rounding into the factors: relative
            // error of 24 lengths from 18000 to 10^6 1.76e-7 in the mean, 1.56e-7
            // now (18000 1.77e-7 -> 1.51e-7).
            const long long col = c0 + cl + a.tw4_c0;
            if constexpr (sizeof(T) == 4) {
                const cx<double> st = tw4<double>(a, (long long)NS * col);
                cx<double> w = tw4<double>(a, (long long)base * col);
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    v[r] = twmul<DIR>(v[r], mk<T>((T)w.x, (T)w.y));
                    if (r + 1 < R) w = cmul(w, st);
                }
            } else {
                const cx<T> st = tw4<T>(a, (long long)NS * col);
#pragma unroll
                for (int r0 = 0; r0 < R; r0 += 4) {
                    cx<T> w = tw4<T>(a, (long long)(base + r0 * NS) * col);
                    v[r0] = twmul<DIR>(v[r0], w);
#pragma unroll
                    for (int r = r0 + 1; r < r0 + 4; ++r)
                        if (r < R) {
                            w = cmul(w, st);
                            v[r] = twmul<DIR>(v[r], w);
                        }
                }
            }
        }
        if (a.scale != 1.0) {
#pragma unroll
            for (int r = 0; r < R; ++r) v[r] = scl(v[r], (T)a.scale);
        }
        cx<T>* q = dst + (long long)base * ond;
        const long long st = (long long)NS * ond;
#pragma unroll
        for (int r = 0; r < R; ++r, q += st) st_out(q, v[r], nt);
    };
    cx<T>* row = COLL ? sm + c : sm + c * P;
    if constexpr (VAR == VAR_4B) {
        cx<T>* rowl = sm + cl * P;
        if (g.npass == 1) {
            // one pass: rows into LDS, then the pass with lanes along c
            if (act)
                for (int n = t; n < g.n; n += TPT) row[n] = src[n];
            __syncthreads();
            auto load_l = [&](auto& v, int j, int NR) __attribute__((always_inline)) {
                constexpr int R = sizeof(v) / sizeof(v[0]);
#pragma unroll
                for (int r = 0; r < R; ++r) v[r] = rowl[j + r * NR];
            };
            mix_pass_any<DIR, true, false, T>(actl, tl, TPT, g.p[0], tw, load_l, store_g, [] {});
            return;
        }
        mix_transform<T, DIR, true>(g, tw, act, t, row, actl, tl, rowl, 1, load_g, store_g);
    } else {
        mix_transform<T, DIR, false>(g, tw, act, t, row, act, t, row, COLL ? G : 1, load_g, store_g);
    }
}

// ---- real rows ---------------------------------------------------------------
// R2C and C2R of rows of 2h reals, h smooth: the h-point transform as in
// k_mix's row layout, the pack and recombination of k_real (kernels.hpp) fused
// into it.  Each thread recombines pairs of bins k and h - k, which share
// their two points and (up to sign and conjugation) their twiddle W_N^k, in
// LDS: after the last pass for R2C, before the first one for C2R.  Before,
// these rows ran the transform and the recombination as two launches with the
// whole intermediate in memory between them; 1920 float32 reals, 17280 rows:
// R2C 0.128 -> 0.052 ms (two launches against one).
struct MixRealArgs {
    MixArgs m;            // in_cd / out_cd: row distances in complex elements of each side
    const void* wk;       // W_N^k, k < h (forward sign)
};

template <typename T, int DIR>
__global__ void __launch_bounds__(MixCfg<T>::THREADS, MixCfg<T>::WAVES) k_mix_real(MixRealArgs g) {
    extern __shared__ unsigned char smraw[];
    cx<T>* sm = (cx<T>*)smraw;
    const KArgs a = g.m.k;
    const int G = g.m.g, TPT = g.m.tpt, tid = threadIdx.x, P = g.m.pitch, H = g.m.n, np = g.m.npass - 1;
    int t;
    const int c = fast_divmod(tid, TPT, g.m.divm, &t);
    const long long cg = (long long)blockIdx.x * G + c;
    const bool act = tid < G * TPT && cg < a.count;
    const cx<T>* __restrict__ src = (const cx<T>*)a.in + cg * a.in_cd;
    cx<T>* __restrict__ dst = (cx<T>*)a.out + cg * a.out_cd;
    const cx<T>* __restrict__ tw = (const cx<T>*)a.tw;
    const cx<T>* __restrict__ wk = (const cx<T>*)g.wk;
    cx<T>* row = sm + c * P;
    const T half = T(0.5), sc = (T)a.scale;
    auto load_s = [&](auto& v, int j, int NR) __attribute__((always_inline)) {
        constexpr int R = sizeof(v) / sizeof(v[0]);
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = row[j + r * NR];
    };
    auto store_s = [&](auto& v, int base, int NS) __attribute__((always_inline)) {
        constexpr int R = sizeof(v) / sizeof(v[0]);
#pragma unroll
        for (int r = 0; r < R; ++r) row[base + r * NS] = v[r];
    };
    auto sync = [] { __syncthreads(); };
    auto none = [] {};
    if constexpr (DIR < 0) {
        auto load_g = [&](auto& v, int j, int NR) __attribute__((always_inline)) {
            constexpr int R = sizeof(v) / sizeof(v[0]);
            const cx<T>* q = src + j;
#pragma unroll
            for (int r = 0; r < R; ++r, q += NR) v[r] = *q;
        };
        mix_pass_any<-1, true, true, T>(act, t, TPT, g.m.p[0], tw, load_g, store_s, none);
        __syncthreads();
        for (int p = 1; p <= np; ++p) {
            mix_pass_any<-1, false, true, T>(act, t, TPT, g.m.p[p], tw + g.m.p[p].twoff, load_s, store_s, sync);
            __syncthreads();
        }
        if (!act) return;
        for (int k = t; 2 * k <= H; k += TPT) {
            const cx<T> A = row[k];
            if (k == 0) {
                dst[0] = mk<T>((A.x + A.y) * sc, T(0));
                dst[H] = mk<T>((A.x - A.y) * sc, T(0));
            } else {
                const cx<T> B = conjx(row[H - k]);
                const cx<T> S2 = scl(A + B, half), D = rot<-1>(cmul(wk[k], scl(A - B, half)));
                dst[k] = scl(S2 + D, sc);
                dst[H - k] = conjx(scl(S2 - D, sc));
            }
        }
    } else {
        if (act) {
#pragma unroll 4
            for (int k = t; 2 * k <= H; k += TPT) {
                cx<T> A = src[k], B = conjx(src[H - k]);
                if (k == 0) { A.y = T(0); B.y = T(0); }
                const cx<T> S2 = scl(A + B, half), D = rot<1>(cmulc(scl(A - B, half), wk[k]));
                row[k] = S2 + D;   // + i conj(W) D
                if (k) row[H - k] = conjx(S2 - D);
            }
        }
        __syncthreads();
        auto store_g = [&](auto& v, int base, int NS) __attribute__((always_inline)) {
            constexpr int R = sizeof(v) / sizeof(v[0]);
            cx<T>* q = dst + base;
#pragma unroll
            for (int r = 0; r < R; ++r, q += NS) *q = scl(v[r], sc);
        };
        if (np == 0) {
            mix_pass_any<1, true, false, T>(act, t, TPT, g.m.p[0], tw, load_s, store_g, none);
            return;
        }
        mix_pass_any<1, true, true, T>(act, t, TPT, g.m.p[0], tw, load_s, store_s, sync);
        __syncthreads();
        for (int p = 1; p < np; ++p) {
            mix_pass_any<1, false, true, T>(act, t, TPT, g.m.p[p], tw + g.m.p[p].twoff, load_s, store_s, sync);
            __syncthreads();
        }
        mix_pass_any<1, false, false, T>(act, t, TPT, g.m.p[np], tw + g.m.p[np].twoff, load_s, store_g, none);
    }
}

}  // namespace afft
