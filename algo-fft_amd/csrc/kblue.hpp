// Lengths with a prime factor above 7 as one cyclic convolution per row, on
// the passes of k_mix (kmix.hpp), all in LDS with one read and one write of
// memory per point: Bluestein's chirp form padded to any 7-smooth M >= 2n - 1,
// and Rader's form for primes n with n - 1 7-smooth, whose convolution has
// n - 1 points and no padding.
//
// A block holds G rows, TPT threads each.  A row goes to LDS, is transformed
// there, multiplied by the filter's spectrum (1/M folded in) while the first
// pass of the inverse transform reads it, and leaves from the last pass
// (Bluestein) or through LDS, where that pass scatters it (Rader).
//
// Bound by the arithmetic and the LDS passes of two transforms of M points,
// so by M.  8192 complex64 rows of 1009 points, where the power-of-two chain
// (k_blue) ran 2048 points: 0.070 -> 0.050 ms; 8172 rows of 2053, 8192 -> 4200 points:
// 0.354 -> 0.191 ms.
#pragma once
#include "kmix.hpp"

namespace afft {

struct MixBlueArgs {
    MixArgs m;                   // M points; in_cd / out_cd, count, scale
    const void* chirp;           // Bluestein: n entries, forward sign
    const void* filt;            // M entries
    const unsigned short* perm;  // Rader: g^q mod n, q < M = n - 1
    int n;
    int inverse;                 // conj(chirp); the filter carries its own direction
};

template <typename T, bool RADER>
__global__ void __launch_bounds__(MixCfg<T>::THREADS, MixCfg<T>::WAVES) k_mix_blue(MixBlueArgs g) {
    extern __shared__ unsigned char smraw[];
    cx<T>* sm = (cx<T>*)smraw;
    const int G = g.m.g, TPT = g.m.tpt, tid = threadIdx.x, M = g.m.n, np = g.m.npass - 1, n = g.n;
    int t;
    const int c = fast_divmod(tid, TPT, g.m.divm, &t);
    const long long cg = (long long)blockIdx.x * G + c;
    const bool act = tid < G * TPT && cg < g.m.k.count;
    const cx<T>* __restrict__ tw = (const cx<T>*)g.m.k.tw;
    const cx<T>* __restrict__ chirp = (const cx<T>*)g.chirp;
    const cx<T>* __restrict__ filt = (const cx<T>*)g.filt;
    const unsigned short* __restrict__ perm = g.perm;
    const cx<T>* __restrict__ src = (const cx<T>*)g.m.k.in + cg * g.m.k.in_cd;
    cx<T>* __restrict__ dst = (cx<T>*)g.m.k.out + cg * g.m.k.out_cd;
    int off = c * g.m.pitch;
    cx<T>* row = sm + off;
    // keeps the compiler from computing every radix's addresses ahead of both
    // transforms, which spills
    auto fresh = [&]() __attribute__((always_inline)) {
        asm volatile("" : "+v"(t), "+v"(off));
        row = sm + off;
    };
    const T sg = g.inverse ? T(-1) : T(1), sc = (T)g.m.k.scale;
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

    if (act) {
        if constexpr (RADER) {
#pragma unroll 4
            for (int i = t; i <= M; i += TPT) row[i] = src[i];
        } else {
#pragma unroll 4
            for (int i = t; i < M; i += TPT) {
                cx<T> y = mk<T>(0, 0);
                if (i < n) {
                    const cx<T> w = chirp[i];
                    y = cmul(src[i], mk<T>(w.x, w.y * sg));
                }
                row[i] = y;
            }
        }
    }
    __syncthreads();
    cx<T> x0 = mk<T>(0, 0), dc = mk<T>(0, 0);
    if constexpr (RADER) {
        if (act && t == 0) x0 = row[0];
        auto load_p = [&](auto& v, int j, int NR) __attribute__((always_inline)) {
            constexpr int R = sizeof(v) / sizeof(v[0]);
#pragma unroll
            for (int r = 0; r < R; ++r) v[r] = row[perm[j + r * NR]];
        };
        mix_pass_any<-1, true, true, T>(act, t, TPT, g.m.p[0], tw, load_p, store_s, sync);
    } else {
        mix_pass_any<-1, true, true, T>(act, t, TPT, g.m.p[0], tw, load_s, store_s, sync);
    }
    __syncthreads();
    for (int p = 1; p <= np; ++p) {
        mix_pass_any<-1, false, true, T>(act, t, TPT, g.m.p[p], tw + g.m.p[p].twoff, load_s, store_s, sync);
        __syncthreads();
    }
    fresh();
    if constexpr (RADER) {
        if (act && t == 0) dc = x0 + row[0];   // bin 0: the sum of the row
    }
    // butterfly 0 of the first pass is thread 0's: adding x[0] to bin 0 adds
    // it to every output
    auto load_f = [&](auto& v, int j, int NR) __attribute__((always_inline)) {
        constexpr int R = sizeof(v) / sizeof(v[0]);
        const cx<T>* f = filt + j;
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = cmul(row[j + r * NR], f[r * NR]);
        if constexpr (RADER) {
            if (j == 0) v[0] = v[0] + x0;
        }
    };
    if constexpr (RADER) {
        // output q is bin g^-q
        auto store_p = [&](auto& v, int base, int NS) __attribute__((always_inline)) {
            constexpr int R = sizeof(v) / sizeof(v[0]);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int q = base + r * NS;
                row[perm[q ? M - q : 0]] = v[r];
            }
        };
        if (np == 0) {
            mix_pass_any<1, true, true, T>(act, t, TPT, g.m.p[0], tw, load_f, store_p, sync);
        } else {
            mix_pass_any<1, true, true, T>(act, t, TPT, g.m.p[0], tw, load_f, store_s, sync);
            __syncthreads();
            for (int p = 1; p < np; ++p) {
                mix_pass_any<1, false, true, T>(act, t, TPT, g.m.p[p], tw + g.m.p[p].twoff, load_s, store_s, sync);
                __syncthreads();
            }
            mix_pass_any<1, false, true, T>(act, t, TPT, g.m.p[np], tw + g.m.p[np].twoff, load_s, store_p, sync);
        }
        if (act && t == 0) row[0] = dc;
        __syncthreads();
        if (act) {
#pragma unroll 4
            for (int i = t; i <= M; i += TPT) dst[i] = scl(row[i], sc);
        }
    } else {
        auto store_g = [&](auto& v, int base, int NS) __attribute__((always_inline)) {
            constexpr int R = sizeof(v) / sizeof(v[0]);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int k = base + r * NS;
                if (k < n) {
                    const cx<T> w = chirp[k];
                    dst[k] = scl(cmul(v[r], mk<T>(w.x, w.y * sg)), sc);
                }
            }
        };
        if (np == 0) {
            mix_pass_any<1, true, false, T>(act, t, TPT, g.m.p[0], tw, load_f, store_g, none);
            return;
        }
        mix_pass_any<1, true, true, T>(act, t, TPT, g.m.p[0], tw, load_f, store_s, sync);
        __syncthreads();
        for (int p = 1; p < np; ++p) {
            mix_pass_any<1, false, true, T>(act, t, TPT, g.m.p[p], tw + g.m.p[p].twoff, load_s, store_s, sync);
            __syncthreads();
        }
        mix_pass_any<1, false, false, T>(act, t, TPT, g.m.p[np], tw + g.m.p[np].twoff, load_s, store_g, none);
    }
}

}  // namespace afft
