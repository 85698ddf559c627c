// In-place runtime-radix Stockham passes of the ragged batch's kernels
// (kragged.hpp): one prime or power-of-two radix per pass.
#pragma once
#include "kernels.hpp"

namespace afft {

// Twiddles w^1 .. w^(R-1) of one butterfly from its k-major table entries
// w[r-1] = w^r.  For complex128, radices 4 and up load w^1, w^2 (and w^4,
// w^8 for radix 8 and 16) and form the other powers as at most two products
// (a few ulps): the table loads of a pass drop from one per point to about
// one per four points for radix 16.  Measured on 512 MiB batches:
// complex128 rows of 3000 points 0.326 -> 0.302 ms (on an earlier row kernel).
// Complex64 passes (tw_apply) load every power as they apply it: the
// products' registers took the 4096-job ragged set from 0.499 to 0.562 ms.
template <int R, typename T, class W>
__device__ __forceinline__ void tw_powers(W w, cx<T> (&ww)[R]) {
    if constexpr (R <= 3) {
#pragma unroll
        for (int r = 1; r < R; ++r) ww[r] = w[r - 1];
    } else if constexpr (R == 4 || R == 5 || R == 7) {
        ww[1] = w[0];
        ww[2] = w[1];
        ww[3] = cmul(ww[1], ww[2]);
        if constexpr (R >= 5) ww[4] = cmul(ww[2], ww[2]);
        if constexpr (R == 7) {
            ww[5] = cmul(ww[4], ww[1]);
            ww[6] = cmul(ww[4], ww[2]);
        }
    } else {
        static_assert(R == 8 || R == 16, "radix");
        ww[1] = w[0];
        ww[2] = w[1];
        ww[4] = w[3];
        ww[3] = cmul(ww[1], ww[2]);
        ww[5] = cmul(ww[1], ww[4]);
        ww[6] = cmul(ww[2], ww[4]);
        ww[7] = cmul(ww[3], ww[4]);
        if constexpr (R == 16) {
            ww[8] = w[7];
#pragma unroll
            for (int r = 9; r < 16; ++r) ww[r] = cmul(ww[r - 8], ww[8]);
        }
    }
}

// v[r] *= w^r (r = 1 .. R-1) for the butterfly whose table entries start at w.
template <int R, int DIR, typename T, class W>
__device__ __forceinline__ void tw_apply(W w, cx<T>* v) {
    if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int r = 1; r < R; ++r) v[r] = twmul<DIR>(v[r], w[r - 1]);
    } else {
        cx<T> ww[R];
        tw_powers<R>(w, ww);
#pragma unroll
        for (int r = 1; r < R; ++r) v[r] = twmul<DIR>(v[r], ww[r]);
    }
}

// One in-place radix-R Stockham pass of a transform of N points with
// N/R <= (16/R) * TT: thread t reads butterflies j = t, t+TT, ... (load(n)),
// applies twiddles and the codelet, and after a barrier of the whole block
// writes output point (j/Ns)*Ns*R + j%Ns + r*Ns (store(k, v)).  Every thread
// of the block calls this; `active` threads do the work.
template <int R, int DIR, typename T, class W, class Load, class Store>
__device__ __forceinline__ void rt_pass_ip(bool active, int t, int TT, int N, int NS, unsigned NSM, W tw, Load load,
                                           Store store) {
    constexpr int MB = (16 + R - 1) / R;
    const int NR = N / R;
    cx<T> v[MB][R];
    if (active) {
#pragma unroll
        for (int b = 0; b < MB; ++b) {
            const int j = t + b * TT;
            if (j < NR) {
#pragma unroll
                for (int r = 0; r < R; ++r) v[b][r] = load(j + r * NR);
                const int k = fast_mod(j, NS, NSM);
                if (NS > 1) tw_apply<R, DIR>(tw + k * (R - 1), v[b]);   // k-major table: k*(R-1) + r-1
                dft<R, DIR, 1>(v[b]);
            }
        }
    }
    __syncthreads();
    if (active) {
#pragma unroll
        for (int b = 0; b < MB; ++b) {
            const int j = t + b * TT;
            if (j < NR) {
                const int k = fast_mod(j, NS, NSM);
                const int base = (j - k) * R + k;
#pragma unroll
                for (int r = 0; r < R; ++r) store(base + r * NS, v[b][r]);
            }
        }
    }
}

template <int DIR, typename T, class W, class Load, class Store>
__device__ __forceinline__ void rt_pass_ip_any(int R, bool active, int t, int TT, int N, int NS, unsigned NSM, W tw,
                                               Load load, Store store) {
    switch (R) {
    case 2: rt_pass_ip<2, DIR, T>(active, t, TT, N, NS, NSM, tw, load, store); break;
    case 3: rt_pass_ip<3, DIR, T>(active, t, TT, N, NS, NSM, tw, load, store); break;
    case 4: rt_pass_ip<4, DIR, T>(active, t, TT, N, NS, NSM, tw, load, store); break;
    case 5: rt_pass_ip<5, DIR, T>(active, t, TT, N, NS, NSM, tw, load, store); break;
    case 7: rt_pass_ip<7, DIR, T>(active, t, TT, N, NS, NSM, tw, load, store); break;
    case 8: rt_pass_ip<8, DIR, T>(active, t, TT, N, NS, NSM, tw, load, store); break;
    case 16: rt_pass_ip<16, DIR, T>(active, t, TT, N, NS, NSM, tw, load, store); break;
    default: {   // radix 1: the copy of a one-point transform
        cx<T> v0 = mk<T>(0, 0);
        if (active && t < N) v0 = load(t);
        __syncthreads();
        if (active && t < N) store(t, v0);
    }
    }
}

}  // namespace afft
