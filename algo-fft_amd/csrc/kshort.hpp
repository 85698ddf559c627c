// Linear convolution of batched rows with a short side, summed directly: for
// up to some 50 to 100 taps the multiply-adds cost less than the LDS passes of three
// transforms (kconv.hpp), and the sums carry less rounding.
//
// A block holds G row pairs, TPT threads each, K consecutive outputs a
// thread (or one tile of TPT*K outputs of a long row).  The taps and the
// tile's stretch of the signal, zero-padded, sit in LDS; a thread reads U
// taps (the same ones in all lanes of a row) and the K + U - 1 points under
// them for K*U products.  K is odd, so the lanes' reads fall on different
// banks; complex128 takes 5 outputs (7 leave 170 registers, two waves a SIMD:
// 4060 rows of 1000 with 33 69 us against 45).  The outputs return through LDS
// for stores along the row.
//
// The products are summed in blocks: U/2 taps in turn, two such sums to U taps,
// four of these to a group, the groups in turn.  One sum over all taps rounds
// alike at every step where the signal hardly varies (a moving average): box
// filters of 33, 96 and 128 taps over constant float32 rows then had a relative
// error of 2.1e-7, 6.3e-7 and 9.8e-7, the transforms 0.96e-7, 0.93e-7 and 1.2e-7, the
// blocks 0.3e-7, 0.3e-7 and 0.12e-7; noise with 33 taps 2.0e-7 by transforms, 1.0e-7
// in one sum, 0.67e-7 in blocks.  In the four types, for four kinds of signals and
// 4 to 128 taps the blocks' error is 0.01 to 0.57 of the transforms'.  They
// cost 3 to 25 % of the time (float32 33 taps 32.8 -> 37.3 us, complex128 128 taps 90 -> 112).
//
// Bound by the multiply-adds and additions (K*U products for K + 2U - 1 LDS
// reads), with few taps by the copy in and out.  16384 float32 rows of 1000 with
// 33: 37 us.  Rounding the taps up to U instead of U / 2 and bounds checks on every
// point of the tile had cost a quarter more.
#pragma once
#include "fft_common.hpp"

namespace afft {

struct ShortConvArgs {
    const void *x, *h;     // signal rows (nx), tap rows (nh)
    void* dst;             // rows of len = nx + nh - 1
    long long nx, len, count;
    int nh, nhp;           // taps, rounded up to U / 2
    int xrev, hrev;        // 1: that side's row is read reversed and conjugated
    int g, tpt, pitch;     // pairs per block, threads per pair, LDS elements per pair
};

template <typename T, bool REAL>
struct ShortCfg {
    using E = std::conditional_t<REAL, T, cx<T>>;
    static constexpr int K = REAL ? 9 : sizeof(T) == 8 ? 5 : 7, U = REAL ? 8 : 4, THREADS = 256;
};

__device__ __forceinline__ float conj_of(float v) { return v; }
__device__ __forceinline__ double conj_of(double v) { return v; }
template <typename T>
__device__ __forceinline__ cx<T> conj_of(cx<T> v) { return conjx(v); }
__device__ __forceinline__ void mac(float& a, float h, float x) { a += h * x; }
__device__ __forceinline__ void mac(double& a, double h, double x) { a += h * x; }
template <typename T>
__device__ __forceinline__ void mac(cx<T>& a, cx<T> h, cx<T> x) {
    a.x += h.x * x.x;
    a.x -= h.y * x.y;
    a.y += h.x * x.y;
    a.y += h.y * x.x;
}
__device__ __forceinline__ float prod(float h, float x) { return h * x; }
__device__ __forceinline__ double prod(double h, double x) { return h * x; }
template <typename T>
__device__ __forceinline__ cx<T> prod(cx<T> h, cx<T> x) { return cmul(h, x); }

template <typename T, bool REAL>
__global__ void __launch_bounds__(256) k_conv_short(ShortConvArgs g) {
    using C = ShortCfg<T, REAL>;
    using E = typename C::E;
    constexpr int K = C::K, U = C::U;
    extern __shared__ unsigned char smraw[];
    const int G = g.g, TPT = g.tpt, tid = threadIdx.x, nhp = g.nhp;
    const int c = tid / TPT, t = tid - c * TPT;
    const long long cg = (long long)blockIdx.x * G + c, o0 = (long long)blockIdx.y * TPT * K;
    const bool act = c < G && cg < g.count;
    E* hs = (E*)smraw + (c < G ? c : 0) * g.pitch;
    E* xs = hs + nhp;
    const int W = TPT * K + nhp - 1;
    if (act) {
        const E* __restrict__ x = (const E*)g.x + cg * g.nx;
        const E* __restrict__ h = (const E*)g.h + cg * g.nh;
        // points lo <= i < hi of the tile lie in the row
        const long long at = o0 - (nhp - 1), end = g.nx - at;
        const int lo = at < 0 ? (int)-at : 0, hi = end < W ? (int)end : W;
        for (int i = t; i < lo; i += TPT) xs[i] = E{};
        if (g.xrev) {
            const E* __restrict__ xp = x + (g.nx - 1 - at);
#pragma unroll 4
            for (int i = lo + t; i < hi; i += TPT) xs[i] = conj_of(xp[-i]);
        } else {
            const E* __restrict__ xp = x + at;
#pragma unroll 8
            for (int i = lo + t; i < hi; i += TPT) xs[i] = xp[i];
        }
        for (int i = hi + t; i < W; i += TPT) xs[i] = E{};
        for (int i = t; i < nhp; i += TPT) {
            E v{};
            if (i < g.nh) v = g.hrev ? conj_of(h[g.nh - 1 - i]) : h[i];
            hs[i] = v;
        }
    }
    __syncthreads();
    E tot[K];
#pragma unroll
    for (int k = 0; k < K; ++k) tot[k] = E{};
    if (act) {
        E acc[K];
        auto step = [&](auto uc, int j) __attribute__((always_inline)) {
            constexpr int V = decltype(uc)::value, H = U / 2;
            const E* w0 = xs + t * K + nhp - j;
            E s[K];
#pragma unroll
            for (int v = H; v <= V; v += H) {   // taps j + v - H .. j + v - 1
                E w[K + H - 1], hh[H], q[K];
#pragma unroll
                for (int m = 0; m < K + H - 1; ++m) w[m] = w0[m - v];
#pragma unroll
                for (int u = 0; u < H; ++u) hh[u] = hs[j + v - H + u];
#pragma unroll
                for (int k = 0; k < K; ++k) q[k] = prod(hh[0], w[k + H - 1]);
#pragma unroll
                for (int u = 1; u < H; ++u)
#pragma unroll
                    for (int k = 0; k < K; ++k) mac(q[k], hh[u], w[k + H - 1 - u]);
#pragma unroll
                for (int k = 0; k < K; ++k) s[k] = v == H ? q[k] : s[k] + q[k];
            }
#pragma unroll
            for (int k = 0; k < K; ++k) acc[k] = acc[k] + s[k];
        };
        int j = 0;
#pragma unroll 1
        do {
#pragma unroll
            for (int k = 0; k < K; ++k) acc[k] = E{};
            const int end = j + 4 * U < nhp ? j + 4 * U : nhp;
#pragma unroll 1
            for (; j + U <= end; j += U) step(std::integral_constant<int, U>{}, j);
            if (j < end) {
                step(std::integral_constant<int, U / 2>{}, j);
                j = end;
            }
#pragma unroll
            for (int k = 0; k < K; ++k) tot[k] = tot[k] + acc[k];
        } while (j < nhp);
    }
    __syncthreads();
    if (act) {
#pragma unroll
        for (int k = 0; k < K; ++k) xs[t * K + k] = tot[k];
    }
    __syncthreads();
    if (act) {
        E* __restrict__ y = (E*)g.dst + cg * g.len + o0;
        const long long left = g.len - o0;
        const int n = left < TPT * K ? (int)left : TPT * K;
#pragma unroll 4
        for (int i = t; i < n; i += TPT) y[i] = xs[i];
    }
}

}  // namespace afft
