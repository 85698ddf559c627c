// Linear convolution and cross-correlation of batched rows in one launch:
// both zero-padded transforms, the product of the spectra, the inverse
// transform and the crop, on the passes of k_mix (kmix.hpp), for padded
// lengths held in LDS.
//
// A block holds G row pairs, TPT threads each, and one LDS buffer of a row
// each: the spectrum of b goes from LDS into the registers of the threads
// that multiply its bins (at most 21 points a thread), then the row of a is
// transformed in its place, multiplied and transformed back.  Real rows of F
// points run as h = F/2 complex points; a thread multiplies pairs of bins k
// and h - k, recombined from and back to the packed form on the fly.
//
// Memory traffic is the inputs and the output.  As six or seven launches
// (pad, pad, R2C, product, C2R, crop) every padded row went through memory
// five times: real rows of 1000 with 33, 16384 pairs: 0.237 -> 0.089 ms;
// bound now by the LDS passes (three transforms of a row per row).
#pragma once
#include "kmix.hpp"

namespace afft {

struct MixConvArgs {
    MixArgs m;             // n = F (complex) or F/2 (real); count = batch
    const void *a, *b;     // rows of na and nb elements
    void* dst;             // rows of len = na + nb - 1 elements
    int na, nb, len;
    const void* wk;        // real: W_F^k, k <= F/4 (forward sign)
    int revconj;           // b[i] read as conj(b[nb-1-i])
};

constexpr int MIX_HOLD = 22;   // spectrum values a thread holds (mix_mb(R) * R <= 21, pairs rounded up)

template <typename T, bool REAL>
__global__ void __launch_bounds__(MixCfg<T>::THREADS, MixCfg<T>::WAVES) k_mix_conv(MixConvArgs g) {
    extern __shared__ unsigned char smraw[];
    cx<T>* sm = (cx<T>*)smraw;
    const int G = g.m.g, TPT = g.m.tpt, tid = threadIdx.x, N = g.m.n, np = g.m.npass - 1;
    int t;
    const int c = fast_divmod(tid, TPT, g.m.divm, &t);
    const long long cg = (long long)blockIdx.x * G + c;
    const bool act = tid < G * TPT && cg < g.m.k.count;
    const cx<T>* __restrict__ tw = (const cx<T>*)g.m.k.tw;
    const cx<T>* __restrict__ wk = (const cx<T>*)g.wk;
    int off = c * g.m.pitch;
    cx<T>* row = sm + off;
    // The compiler would compute every radix's addresses once, ahead of the
    // transforms (300-450 spilled registers): hide what they come from.
    auto fresh = [&]() __attribute__((always_inline)) {
        asm volatile("" : "+v"(t), "+v"(off));
        row = sm + off;
    };
    const T half = T(0.5), sc = (T)g.m.k.scale;
    const int len = g.len;
    const bool revconj = g.revconj;
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
    cx<T> hold[MIX_HOLD];

#pragma unroll 1
    for (int side = 0; side < 2; ++side) {   // the row of b, then that of a
        fresh();
        const long long n = side ? g.na : g.nb;
        // zero-padded into LDS first: reading memory inside the first pass,
        // with its bounds, spilled 390-500 registers
        if (act) {
            if constexpr (REAL) {
                const T* __restrict__ x = (const T*)(side ? g.a : g.b) + cg * n;
#pragma unroll 4
                for (int m = t; m < N; m += TPT)
                    row[m] = mk<T>(2 * m < n ? x[2 * m] : T(0), 2 * m + 1 < n ? x[2 * m + 1] : T(0));
            } else {
                const cx<T>* __restrict__ x = (const cx<T>*)(side ? g.a : g.b) + cg * n;
                const bool rc = !side && revconj;
#pragma unroll 4
                for (int m = t; m < N; m += TPT) {
                    cx<T> y = mk<T>(0, 0);
                    if (m < n) y = rc ? conjx(x[n - 1 - m]) : x[m];
                    row[m] = y;
                }
            }
        }
        __syncthreads();
        mix_pass_any<-1, true, true, T>(act, t, TPT, g.m.p[0], tw, load_s, store_s, sync);
        __syncthreads();
        for (int p = 1; p <= np; ++p) {
            mix_pass_any<-1, false, true, T>(act, t, TPT, g.m.p[p], tw + g.m.p[p].twoff, load_s, store_s, sync);
            __syncthreads();
        }
        if (!side) {
            if constexpr (REAL) {
#pragma unroll
                for (int i = 0; i < MIX_HOLD / 2; ++i) {
                    const int k = t + i * TPT;
                    if (act && 2 * k <= N) {
                        hold[2 * i] = row[k];
                        hold[2 * i + 1] = row[k ? N - k : 0];
                    }
                }
            } else {
#pragma unroll
                for (int i = 0; i < MIX_HOLD; ++i) {
                    const int k = t + i * TPT;
                    if (act && k < N) hold[i] = row[k];
                }
            }
            __syncthreads();
        }
    }
    fresh();
    if constexpr (REAL) {
#pragma unroll
        for (int i = 0; i < MIX_HOLD / 2; ++i) {
            const int k = t + i * TPT;
            if (act && 2 * k <= N) {
                const cx<T> A = row[k];
                if (k == 0) {
                    // bins 0 and N are real: their products, packed back
                    const cx<T> B = hold[0];
                    const T p0 = (A.x + A.y) * (B.x + B.y), pn = (A.x - A.y) * (B.x - B.y);
                    row[0] = mk<T>((p0 + pn) * half, (p0 - pn) * half);
                } else {
                    const cx<T> A2 = conjx(row[N - k]), B = hold[2 * i], B2 = conjx(hold[2 * i + 1]), w = wk[k];
                    const cx<T> SA = scl(A + A2, half), DA = rot<-1>(cmul(w, scl(A - A2, half)));
                    const cx<T> SB = scl(B + B2, half), DB = rot<-1>(cmul(w, scl(B - B2, half)));
                    // bins k and N - k of either side: S + D and conj(S - D)
                    const cx<T> P = cmul(SA + DA, SB + DB), P2 = cmul(SA - DA, SB - DB);   // P2 = conj(bin N - k)
                    const cx<T> S = scl(P + P2, half), D = rot<1>(cmulc(scl(P - P2, half), w));
                    row[k] = S + D;
                    row[N - k] = conjx(S - D);
                }
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < MIX_HOLD; ++i) {
            const int k = t + i * TPT;
            if (act && k < N) row[k] = cmul(row[k], hold[i]);
        }
    }
    __syncthreads();
    fresh();
    auto store_g = [&](auto& v, int base, int NS) __attribute__((always_inline)) {
        constexpr int R = sizeof(v) / sizeof(v[0]);
        if constexpr (REAL) {
            T* __restrict__ y = (T*)g.dst + cg * len;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int i = 2 * (base + r * NS);
                if (i < len) y[i] = v[r].x * sc;
                if (i + 1 < len) y[i + 1] = v[r].y * sc;
            }
        } else {
            cx<T>* __restrict__ y = (cx<T>*)g.dst + cg * len;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int k = base + r * NS;
                if (k < len) y[k] = scl(v[r], sc);
            }
        }
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

}  // namespace afft
