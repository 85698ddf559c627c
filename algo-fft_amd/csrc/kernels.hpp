// Batched LDS-resident FFT kernels built on the compile-time Stockham core.
//
// Addressing of transform c (blockIdx.x*TPB + local c) in slice blockIdx.y:
//   element n at  base + blockIdx.y*bd + c*cd + n*nd      (separately for in/out)
// Variants:
//   VAR_ROW  each transform contiguous (nd = 1): ForwardBatch, N-D last axis
//   VAR_COL  TPB adjacent columns (cd = 1), element stride nd: strided plans,
//            N-D outer axes
//   VAR_4A   VAR_COL + four-step twiddle W_L^{k*c} on the outputs (L = N*count)
//   VAR_4B   rows in (nd = 1), outputs scattered as columns (cd = 1): the
//            transposing second pass of the four-step transform.  Its last
//            pass runs with lanes along c, so both sides stay coalesced
#pragma once
#include <utility>

#include "fft_core.hpp"

namespace afft {

enum { VAR_ROW = 0, VAR_COL = 1, VAR_4A = 2, VAR_4B = 3, VAR_COUNT = 4, VAR_BLUE = 4, VAR_REAL = 5, VAR_BLUEMID = 6 };

struct KArgs {
    const void* in;
    void* out;
    const void* tw;          // per-pass twiddle table of the schedule
    long long count;         // transforms along c
    long long in_cd, out_cd;
    long long in_nd, out_nd;
    long long in_bd, out_bd;
    double scale;            // applied when != 1 (inverse 1/N)
    const void* tw4_lo;      // four-step: W_L^m = hi[m >> sh] * lo[m & (2^sh-1)]
    const void* tw4_hi;
    int tw4_shift;
    long long tw4_L;
    long long tw4_c0;        // column index offset of this launch
    int tw4_by_y;            // 1: the four-step column index is blockIdx.y, not c
    // Bluestein fusion on the column passes (runtime, uniform per launch):
    //   FUSE_CHIRP_IN (VAR_4A): x[n] * chirp[n] for n < flen, zero beyond
    //   FUSE_CROP_OUT (VAR_COL): y[k] * fvec[k] stored only for k < flen
    int fuse;
    int fconj;               // use conj(fvec)
    const void* fvec;
    long long flen;
    int nt;                  // NT_STORE / NT_LOAD: non-temporal output stores / input loads
    int xcd;                 // column layouts of k_fft: blocks in XCD order (xcd_block)
};

enum { FUSE_NONE = 0, FUSE_CHIRP_IN = 1, FUSE_CROP_OUT = 2 };

template <typename T>
__device__ __forceinline__ cx<T> fvec_at(const void* f, long long i, int conj) {
    cx<T> w = ((const cx<T>*)f)[i];
    return conj ? conjx(w) : w;
}

template <typename T, int N>
struct PadFor {
    static constexpr int value = N >= 32 ? (sizeof(T) == 4 ? 4 : 3) : 0;
};

template <typename T, class S, int E, int TPB, int VAR>
struct KCfg {
    static constexpr int N = S::N;
    static constexpr int TT = N / E;
    static constexpr int THREADS = TPB * TT;
    static constexpr bool ROWL = (VAR == VAR_ROW || VAR == VAR_4B);
    static constexpr int PADSH = PadFor<T, N>::value;
    static constexpr int LDS_ELEMS = S::P > 1 || VAR == VAR_4B
                                         ? (ROWL ? TPB * LdsRow<N, PADSH>::SLAB : TPB * N)
                                         : 1;
    // Whether k_fft has a second form of this kernel with planar exchanges
    // (planar_exchange): 64 KiB of LDS a block instead of 128, so that one block
    // loads and stores while the other computes.
    // Taken from two blocks a CU on (make_step).  complex128 rows of 8192
    // points, 4096 rows 0.228 -> 0.188 ms, 512 33.7 -> 28.4 us; columns of 1024
    // complex64 points, 64 x 1024 x 1000 0.457 -> 0.431 ms, 16 real images of 1024 x
    // 1024 63 -> 60 us; of 512 complex128, 16 x 512 x 500 52 -> 48 us, 1,000,003 points x
    // 8 0.383 -> 0.365 ms (line-aligned pitches come out even).
    // Other kernels of that size lose by the barriers: complex64 rows of 16384
    // 0.238 -> 0.272, transposing rows (2^20 complex64 0.448 -> 0.479), four-step
    // columns (2^18 complex128 0.208 -> 0.215, 2^22 complex64 0.566 -> 0.602), columns of
    // 512 (0.566 -> 0.570) and 2048 complex64 (0.433 -> 0.441).
    static constexpr bool PLANAR = sizeof(T) == 4 ? VAR == VAR_COL && N == 1024
                                                  : (VAR == VAR_ROW && N == 8192) || (VAR == VAR_COL && N == 512);
};

// Forward-sign W_L^m from the two-level table; callers conjugate for DIR=+1.
template <typename T>
__device__ __forceinline__ cx<T> tw4(const KArgs& a, long long m) {
    const cx<T>* lo = (const cx<T>*)a.tw4_lo;
    const cx<T>* hi = (const cx<T>*)a.tw4_hi;
    const long long mask = (1LL << a.tw4_shift) - 1;
    return cmul(lo[m & mask], hi[m >> a.tw4_shift]);
}

// The work item of this block for neighbouring items on one XCD: consecutive
// blocks go to the 8 XCDs (each with its own L2) in turn; the result is the
// item of the block's position within its XCD's share (a bijection of the
// grid).
__device__ __forceinline__ void xcd_block(unsigned* bx, unsigned* by) {
    constexpr unsigned XCDS = 8;
    const unsigned tot = gridDim.x * gridDim.y, lin = *by * gridDim.x + *bx;
    const unsigned q = tot / XCDS, r = tot % XCDS, x = lin % XCDS;
    const unsigned nl = x * q + (x < r ? x : r) + lin / XCDS;
    *by = nl / gridDim.x;
    *bx = nl - *by * gridDim.x;
}

template <typename T, class S, int E, int TPB, int VAR, int DIR, bool PLANAR = false>
__global__ void __launch_bounds__((KCfg<T, S, E, TPB, VAR>::THREADS)) k_fft(KArgs a) {
    using C = KCfg<T, S, E, TPB, VAR>;
    constexpr int N = S::N;
    constexpr int TT = C::TT;
    using Slot = std::conditional_t<PLANAR, T, cx<T>>;
    __shared__ Slot lds[C::LDS_ELEMS];
    const int tid = threadIdx.x;
    int c, t;
    if constexpr (C::ROWL) { c = tid / TT; t = tid % TT; }
    else { c = tid % TPB; t = tid / TPB; }
    unsigned bx = blockIdx.x, by = blockIdx.y;
    if constexpr (VAR != VAR_ROW)
        if (a.xcd) xcd_block(&bx, &by);
    const long long cg = (long long)bx * TPB + c;
    const bool act = cg < a.count;
    const cx<T>* __restrict__ in = (const cx<T>*)a.in + (long long)by * a.in_bd;
    const cx<T>* __restrict__ tw = (const cx<T>*)a.tw;
    cx<T> v[E];

    if constexpr (VAR == VAR_ROW) {
        const cx<T>* src = in + cg * a.in_cd;
        if (a.nt & NT_LOAD) {
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = act ? ld_nt(src + t + TT * e) : mk<T>(0, 0);
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = act ? src[t + TT * e] : mk<T>(0, 0);
        }
    } else if constexpr (VAR == VAR_4B) {
        const cx<T>* src = in + cg * a.in_cd;
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = act ? src[t + TT * e] : mk<T>(0, 0);
    } else if (VAR == VAR_4A && a.fuse == FUSE_CHIRP_IN) {
        // element n of the padded sequence sits at offset n of a unit-stride row
        const long long nd = a.in_nd;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const long long n = cg + (long long)(t + TT * e) * nd;
            v[e] = (act && n < a.flen) ? cmul(in[n], fvec_at<T>(a.fvec, n, a.fconj)) : mk<T>(0, 0);
        }
    } else {
        const cx<T>* src = in + cg;
        const long long nd = a.in_nd;
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = act ? src[(long long)(t + TT * e) * nd] : mk<T>(0, 0);
    }

    // VAR_4B stores with lanes along c: transform c2, thread t2 of it
    const int c2 = tid % TPB, t2 = tid / TPB;
    if constexpr (PLANAR && C::ROWL) {
        core_planar<T, S, E, DIR, 0>(v, lds, t, tw, LdsRow<N, C::PADSH>(c));
    } else if constexpr (PLANAR) {
        core_planar<T, S, E, DIR, 0>(v, lds, t, tw, LdsCol<TPB>(c));
    } else if constexpr (VAR == VAR_4B && S::P > 1) {
        // The last pass already runs with lanes along c: without a trip
        // through LDS of its own for the store, 512 MiB of complex64 2^20
        // 0.464 -> 0.448 ms, 65536 0.362 -> 0.358, 2^22 0.583 -> 0.566,
        // complex128 2^20 0.457 -> 0.441.
        core_turn<T, S, E, DIR>(v, lds, t, tw, LdsRow<N, C::PADSH>(c), t2, LdsRow<N, C::PADSH>(c2));
    } else if constexpr (C::ROWL) {
        LdsRow<N, C::PADSH> li(c);
        // one row per block of at most 256 threads: twiddle loads ahead of
        // each pass's barrier.  Measured on 512 MiB batches: complex64
        // N=4096 0.182 -> 0.177 ms, complex128 N=4096 0.189 -> 0.187 ms;
        // with several rows per block (N=256), in the four-step passes and
        // in the 512- and 1024-thread rows (complex128 8192, complex64
        // 16384) it lost 1-2 %.
        core<T, S, E, DIR, false, VAR == VAR_ROW && TPB == 1 && N / E <= 256>(v, lds, t, tw, li);
    } else {
        LdsCol<TPB> li(c);
        core<T, S, E, DIR>(v, lds, t, tw, li);
    }

    if constexpr (VAR == VAR_4A) {
        const long long col = (a.tw4_by_y ? (long long)by : cg) + a.tw4_c0;
        // W_L^{k*col} for k = t + TT*e (k < N and col < L/N, so k*col < L
        // needs no reduction).  Lanes differ in col, so every table load
        // gathers from scattered lines: look up every fourth e and step
        // between them by W_L^{TT*col}, at most three products from a
        // table value (10 table loads per thread instead of 2E).
        if constexpr (E % 4 == 0) {
            const cx<T> st = tw4<T>(a, (long long)TT * col);
#pragma unroll
            for (int e0 = 0; e0 < E; e0 += 4) {
                cx<T> w = tw4<T>(a, (long long)(t + TT * e0) * col);
                v[e0] = twmul<DIR>(v[e0], w);
#pragma unroll
                for (int e = e0 + 1; e < e0 + 4; ++e) {
                    w = cmul(w, st);
                    v[e] = twmul<DIR>(v[e], w);
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = twmul<DIR>(v[e], tw4<T>(a, (long long)(t + TT * e) * col));
        }
    }
    if (a.scale != 1.0) {
        const T s = (T)a.scale;
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = scl(v[e], s);
    }

    cx<T>* __restrict__ out = (cx<T>*)a.out + (long long)by * a.out_bd;
    if constexpr (VAR == VAR_ROW) {
        if (act) {
            cx<T>* dst = out + cg * a.out_cd;
#pragma unroll
            for (int e = 0; e < E; ++e) st_out(dst + t + TT * e, v[e], a.nt);
        }
    } else if constexpr (VAR == VAR_COL || VAR == VAR_4A) {
        if (act) {
            cx<T>* dst = out + cg;
            const long long nd = a.out_nd;
            if (VAR == VAR_COL && a.fuse == FUSE_CROP_OUT) {
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const long long k = cg + (long long)(t + TT * e) * nd;
                    if (k < a.flen) out[k] = cmul(v[e], fvec_at<T>(a.fvec, k, a.fconj));
                }
            } else {
#pragma unroll
                for (int e = 0; e < E; ++e) st_out(dst + (long long)(t + TT * e) * nd, v[e], a.nt);
            }
        }
    } else {
        if constexpr (S::P == 1) {   // one pass: re-map through LDS
            LdsRow<N, C::PADSH> li(c), li2(c2);
            __syncthreads();
#pragma unroll
            for (int e = 0; e < E; ++e) lds[li(t + TT * e)] = v[e];
            __syncthreads();
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = lds[li2(t2 + TT * e)];
        }
        const long long cg2 = (long long)bx * TPB + c2;
        if (cg2 < a.count) {
            const long long nd = a.out_nd;
#pragma unroll
            for (int e = 0; e < E; ++e) st_out(out + cg2 + (long long)(t2 + TT * e) * nd, v[e], a.nt);
        }
    }
}

// ---- fused Bluestein chain for a padded length M held in LDS ---------------
// a[n] = x[n]*chirp[n] (n < N, zero to M), A = FFT_M(a), A *= F (the filter
// spectrum with 1/M folded in), y = IFFT_M(A), X[k] = y[k]*chirp[k]*scale.
// The inverse transform uses conj(chirp) and its own filter.  Both FFTs run
// on the register/LDS core; one global read and one global write per point
// (plan_bluestein.go:7-58, internal/kernels/bluestein.go:39-77).
struct BArgs {
    const void* in;
    void* out;
    const void* tw;       // schedule twiddles of M
    const void* chirp;    // N entries, forward sign
    const void* filt;     // M entries
    long long count;
    long long in_cd, out_cd;
    long long nlog;
    double scale;
};

template <typename T, class S, int E, int TPB, int DIR>
__global__ void __launch_bounds__((KCfg<T, S, E, TPB, VAR_ROW>::THREADS)) k_blue(BArgs a) {
    using C = KCfg<T, S, E, TPB, VAR_ROW>;
    constexpr int TT = C::TT;
    __shared__ cx<T> lds[C::LDS_ELEMS];
    const int tid = threadIdx.x;
    const int c = tid / TT, t = tid % TT;
    const long long cg = (long long)blockIdx.x * TPB + c;
    const bool act = cg < a.count;
    const cx<T>* __restrict__ src = (const cx<T>*)a.in + cg * a.in_cd;
    const cx<T>* __restrict__ chirp = (const cx<T>*)a.chirp;
    const cx<T>* __restrict__ filt = (const cx<T>*)a.filt;
    const cx<T>* __restrict__ tw = (const cx<T>*)a.tw;
    cx<T> v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int n = t + TT * e;
        v[e] = (act && n < a.nlog) ? twmul<DIR>(src[n], chirp[n]) : mk<T>(0, 0);
    }
    LdsRow<S::N, C::PADSH> li(c);
    core<T, S, E, -1>(v, lds, t, tw, li);
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = cmul(v[e], filt[t + TT * e]);
    core<T, S, E, 1, true>(v, lds, t, tw, li);
    if (act) {
        cx<T>* dst = (cx<T>*)a.out + cg * a.out_cd;
        const T sc = (T)a.scale;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int n = t + TT * e;
            if (n < a.nlog) dst[n] = scl(twmul<DIR>(v[e], chirp[n]), sc);
        }
    }
}

// Middle pass of a Bluestein chain whose M = m1 * m2 is beyond LDS, between
// the column passes over m1: row k1 of the forward transform's m1 x m2
// intermediate runs its FFT over n2, the product with the filter (stored
// row-major as [k1][k2] for k = k1 + m1*k2), the inverse FFT over k2 and the
// inverse twiddle W_M^{-k1*n2}, in place and contiguous.  The spectrum is
// never put into natural order, so the chain has three passes and no
// transposing store (as four four-step passes: complex128 1,000,003 points x 8
// 0.586 -> 0.384 ms, complex64 100,003 x 64 0.235 -> 0.159, complex128 10,007 x
// 400 0.359 -> 0.228).  Bound by the column passes' access pattern.
// in_cd / out_cd: m2; fvec: the filter, 1/M folded in.
template <typename T, class S, int E, int TPB>
__global__ void __launch_bounds__((KCfg<T, S, E, TPB, VAR_ROW>::THREADS)) k_bluemid(KArgs a) {
    using C = KCfg<T, S, E, TPB, VAR_ROW>;
    constexpr int TT = C::TT;
    __shared__ cx<T> lds[C::LDS_ELEMS];
    const int tid = threadIdx.x;
    const int c = tid / TT, t = tid % TT;
    const long long cg = (long long)blockIdx.x * TPB + c;
    const bool act = cg < a.count;
    const cx<T>* __restrict__ src = (const cx<T>*)a.in + (long long)blockIdx.y * a.in_bd + cg * a.in_cd;
    const cx<T>* __restrict__ filt = (const cx<T>*)a.fvec + cg * a.in_cd;
    const cx<T>* __restrict__ tw = (const cx<T>*)a.tw;
    cx<T> v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = act ? src[t + TT * e] : mk<T>(0, 0);
    LdsRow<S::N, C::PADSH> li(c);
    core<T, S, E, -1>(v, lds, t, tw, li);
    if (act) {
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = cmul(v[e], filt[t + TT * e]);
    }
    core<T, S, E, 1, true>(v, lds, t, tw, li);
    if (act) {
        cx<T>* dst = (cx<T>*)a.out + (long long)blockIdx.y * a.out_bd + cg * a.out_cd;
        const cx<T> st = tw4<T>(a, (long long)TT * cg);
        cx<T> w = mk<T>(1, 0);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            w = e % 4 == 0 ? tw4<T>(a, (long long)(t + TT * e) * cg) : cmul(w, st);
            dst[t + TT * e] = cmulc(v[e], w);
        }
    }
}

// ---- real transforms: pack/unpack fused into the first/last pass --------------
// R2C (PlanRealT.forwardSingle, plan_real_generic.go:142-228): the N reals of
// a row are read as h = N/2 complex points z[m] = x[2m] + i x[2m+1]; after the
// h-point FFT Z sits in LDS and each thread recombines its bins
//   X[k] = ½(A + B) - ½ i W_N^k (A - B),   A = Z[k], B = conj(Z[h-k])
// (the reference's X = A - U[k](A - B) with U[k] = ½(1 + i W_N^k)), with
// X[0] = Re Z0 + Im Z0 and X[h] = Re Z0 - Im Z0.
// C2R (inverseSingle :289-355 with RepackInverse, real_repack.go:49-75):
// the h+1 bins go through LDS, each thread forms
//   Z[k] = ½(A + B) + ½ i conj(W_N^k) (A - B),   A = X[k], B = conj(X[h-k])
// (imaginary parts of X[0], X[h] ignored, as the reference uses only their
// real parts), then the inverse h-point FFT scaled by 1/h gives x as pairs.
struct RArgs {
    const void* in;
    void* out;
    const void* tw;       // schedule twiddles of h
    const void* wk;       // W_N^k, k < h (forward sign)
    long long count;
    long long in_d, out_d;   // per-row distance in complex elements of each side
    double scale;
};

template <typename T, class S, int E, int TPB, int DIR>
__global__ void __launch_bounds__((KCfg<T, S, E, TPB, VAR_ROW>::THREADS)) k_real(RArgs a) {
    using C = KCfg<T, S, E, TPB, VAR_ROW>;
    constexpr int H = S::N;
    constexpr int TT = C::TT;
    using L = LdsRow<H, C::PADSH>;
    __shared__ cx<T> lds[TPB * L::SLAB];
    const int tid = threadIdx.x;
    const int c = tid / TT, t = tid % TT;
    const long long cg = (long long)blockIdx.x * TPB + c;
    const bool act = cg < a.count;
    const cx<T>* __restrict__ src = (const cx<T>*)a.in + cg * a.in_d;
    cx<T>* __restrict__ dst = (cx<T>*)a.out + cg * a.out_d;
    const cx<T>* __restrict__ wk = (const cx<T>*)a.wk;
    const T half = T(0.5);
    const T sc = (T)a.scale;
    L li(c);
    cx<T> v[E];
    if constexpr (DIR < 0) {
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = act ? src[t + TT * e] : mk<T>(0, 0);
        core<T, S, E, -1>(v, lds, t, (const cx<T>*)a.tw, li);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; ++e) lds[li(t + TT * e)] = v[e];
        __syncthreads();
        if (act) {
            // W_N^k for k = t + TT*e: a table value every fourth e and the
            // step W_N^TT in between (at most three products).  Measured on
            // float32 R2C 4096 x 32768: 0.230 -> 0.200 ms against a table
            // load per bin; C2R 512^3 0.788 -> 0.765 ms.
            const cx<T> st = wk[TT];
            cx<T> w = mk<T>(1, 0);
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int k = t + TT * e;
                w = e % 4 == 0 ? wk[k] : cmul(w, st);
                const cx<T> A = lds[li(k)];
                if (k == 0) {
                    dst[0] = mk<T>((A.x + A.y) * sc, T(0));
                    dst[H] = mk<T>((A.x - A.y) * sc, T(0));
                } else {
                    const cx<T> B = conjx(lds[li(H - k)]);
                    const cx<T> S2 = scl(A + B, half), D = scl(A - B, half);
                    const cx<T> X = S2 + rot<-1>(cmul(w, D));
                    dst[k] = scl(X, sc);
                }
            }
        }
    } else {
        // every load of the row in flight at once: as a loop of load and LDS
        // store, 512 float32 reals x 262144 took 0.279 ms instead of 0.185,
        // 4096 x 32768 0.300 instead of 0.202 (two loads per point, without
        // the trip through LDS: 0.207 and 0.215)
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = act ? src[t + TT * e] : mk<T>(0, 0);
        const cx<T> xh = act && t == 0 ? src[H] : mk<T>(0, 0);
#pragma unroll
        for (int e = 0; e < E; ++e) lds[li(t + TT * e)] = v[e];
        if (t == 0) lds[li(H)] = xh;
        __syncthreads();
        const cx<T> st = wk[TT];
        cx<T> w = mk<T>(1, 0);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = t + TT * e;
            w = e % 4 == 0 ? wk[k] : cmul(w, st);
            cx<T> A = lds[li(k)];
            cx<T> B = conjx(lds[li(H - k)]);
            if (k == 0) { A.y = T(0); B.y = T(0); }
            const cx<T> S2 = scl(A + B, half), D = scl(A - B, half);
            v[e] = S2 + rot<1>(cmulc(D, w));   // + i conj(W) D
        }
        core<T, S, E, 1, true>(v, lds, t, (const cx<T>*)a.tw, li);
        if (act) {
#pragma unroll
            for (int e = 0; e < E; ++e) dst[t + TT * e] = scl(v[e], sc);
        }
    }
}

// Stand-alone recombination for the sizes whose h-point FFT runs as its own
// plan step: in = Z (h complex per row), out = X (h+1 per row) for R2C;
// in = X, out = Z for C2R.  One thread per bin.
struct RPArgs {
    const void* in;
    void* out;
    const void* wk;
    long long rows, h;
    long long in_d, out_d;
    double scale;
};
template <typename T, int DIR>
__global__ void __launch_bounds__(256) k_rpost(RPArgs a) {
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long per = DIR < 0 ? a.h + 1 : a.h;
    if (idx >= a.rows * per) return;
    const long long r = idx / per, k = idx - r * per;
    const cx<T>* in = (const cx<T>*)a.in + r * a.in_d;
    cx<T>* out = (cx<T>*)a.out + r * a.out_d;
    const cx<T>* wk = (const cx<T>*)a.wk;
    const T half = T(0.5), sc = (T)a.scale;
    if constexpr (DIR < 0) {
        if (k == 0 || k == a.h) {
            const cx<T> z = in[0];
            out[k] = mk<T>((k == 0 ? z.x + z.y : z.x - z.y) * sc, T(0));
            return;
        }
        const cx<T> A = in[k], B = conjx(in[a.h - k]);
        const cx<T> S2 = scl(A + B, half), D = scl(A - B, half);
        out[k] = scl(S2 + rot<-1>(cmul(wk[k], D)), sc);
    } else {
        cx<T> A = in[k], B = conjx(in[a.h - k]);
        if (k == 0) { A.y = T(0); B.y = T(0); }
        const cx<T> S2 = scl(A + B, half), D = scl(A - B, half);
        out[k] = scl(S2 + rot<1>(cmulc(D, wk[k])), sc);
    }
}

// Strided 2-D copy: element i of line c from in[c*in_cd + i*in_nd] to
// out[c*out_cd + i*out_nd].  Used for length-1 axes and to gather strided
// lines into contiguous rows (and scatter them back) for the paths that need
// unit stride.
struct CopyArgs {
    const void* in;
    void* out;
    long long lines, len;
    long long in_cd, in_nd, out_cd, out_nd;
    double scale;
};
template <typename T>
__global__ void __launch_bounds__(256) k_copy(CopyArgs a) {
    const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= a.lines * a.len) return;
    const long long c = idx / a.len, i = idx - c * a.len;
    cx<T> v = ((const cx<T>*)a.in)[c * a.in_cd + i * a.in_nd];
    if (a.scale != 1.0) v = scl(v, (T)a.scale);
    ((cx<T>*)a.out)[c * a.out_cd + i * a.out_nd] = v;
}

// ---- registry ----------------------------------------------------------------
enum { KIND_FFT = 0, KIND_BLUE = 1, KIND_REAL = 2 };

struct KernelInfo {
    const void* fn;
    const void* planar;   // k_fft with planar exchanges, or null
    int kind;       // KIND_FFT (k_fft) or KIND_BLUE (k_blue)
    int prec;       // 0 = complex64, 1 = complex128
    int n;
    int var;
    int dir;        // -1 forward, +1 inverse
    int e;          // points per thread
    int tpb;        // transforms per block
    int threads;
    int lds_bytes;
    int nrad;
    int rad[8];
};

void register_kernel(const KernelInfo& k);

template <typename T, class S, int E, int TPB, int VAR, int DIR>
struct Registrar {
    Registrar() {
        using C = KCfg<T, S, E, TPB, (VAR >= VAR_BLUE ? VAR_ROW : VAR)>;
        KernelInfo k{};
        if constexpr (VAR == VAR_BLUE) {
            k.fn = (const void*)&k_blue<T, S, E, TPB, DIR>;
            k.kind = KIND_BLUE;
        } else if constexpr (VAR == VAR_BLUEMID) {
            k.fn = (const void*)&k_bluemid<T, S, E, TPB>;   // one kernel for both plan directions
            k.kind = KIND_FFT;
        } else if constexpr (VAR == VAR_REAL) {
            k.fn = (const void*)&k_real<T, S, E, TPB, DIR>;
            k.kind = KIND_REAL;
        } else {
            k.fn = (const void*)&k_fft<T, S, E, TPB, VAR, DIR>;
            if constexpr (C::PLANAR) k.planar = (const void*)&k_fft<T, S, E, TPB, VAR, DIR, true>;
            k.kind = KIND_FFT;
        }
        k.prec = sizeof(T) == 4 ? 0 : 1;
        k.n = S::N;
        k.var = VAR;
        k.dir = DIR;
        k.e = E;
        k.tpb = TPB;
        k.threads = C::THREADS;
        k.lds_bytes = C::LDS_ELEMS * (int)sizeof(cx<T>);
        k.nrad = S::P;
        for (int i = 0; i < S::P; ++i) k.rad[i] = S::rad[i];
        register_kernel(k);
    }
};

}  // namespace afft
