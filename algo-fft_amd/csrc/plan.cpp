// Planner and executor: turns a plan descriptor into a list of kernel
// launches (steps) and runs them.
//
// Size routing (cf. the reference's planner.go:43-78, which picks codelets,
// Stockham, six-step or Bluestein for a CPU):
//   power of two <= LDS capacity (16384 c64 / 8192 c128)  one LDS pass; rows of 16 points to
//                                                         512 bytes and many long columns
//                                                         on the runtime radices
//   power of two above it                                 four-step: column pass with
//                                                         fused twiddle, then a row pass
//                                                         whose store transposes
//   2/3/5/7-smooth                                        runtime radices (k_mix): one pass
//                                                         held in LDS, else four-step
//   anything else (blue_route)                            one launch: Rader's form, or
//                                                         Bluestein's padded to a smooth
//                                                         length or a power of two; where
//                                                         LDS does not hold it, or few
//                                                         rows would leave the chip idle,
//                                                         Bluestein's in three passes
// How many transforms a plan has decides too: launch shapes, Rader or padded
// form and planar exchanges follow it, so the last bits of a transform may
// differ between plans of different batches (never between runs of one plan).
#include <algorithm>
#include <cstdlib>
#include <cstring>

#include <cmath>
#include <complex>
#include <map>
#include <memory>
#include <tuple>

#include "afft_internal.hpp"
#include "kblue.hpp"

namespace afft {

Plan::~Plan() {
    if (ctx) (void)hipSetDevice(ctx->device);
    for (void* q : owned) (void)hipFree(q);
    for (void*& t : tmp)
        if (t) (void)hipFree(t);
    if (stage_in) (void)hipFree(stage_in);
    if (stage_out) (void)hipFree(stage_out);
    if (full) (void)hipFree(full);
    if (pipe) destroy_host_pipe(pipe);
    if (ws_done) (void)hipEventDestroy(ws_done);
    if (stream) (void)hipStreamDestroy(stream);
}

static bool is_pow2(int64_t n) { return n > 0 && (n & (n - 1)) == 0; }
static int ilog2(int64_t n) {
    int l = 0;
    while ((1LL << l) < n) ++l;
    return l;
}

// Upload a host table, owned by the plan.
int upload_table(Plan& p, const void* host, size_t bytes, const void** dev) {
    void* d = nullptr;
    AFFT_HIP(hipMalloc(&d, bytes ? bytes : 16));
    p.owned.push_back(d);
    if (bytes) AFFT_HIP(hipMemcpy(d, host, bytes, hipMemcpyHostToDevice));
    *dev = d;
    return AFFT_OK;
}

// Twiddle table of a radix schedule: for pass i >= 1 with
// Ns = rad[0]*...*rad[i-1] and radix R: entries W_{Ns*R}^{k*r}, k < Ns,
// 1 <= r < R, stored r-major (entry (r-1)*Ns + k), so the lanes of a pass,
// which hold consecutive k, load consecutive entries.  Generated in FP64 and
// rounded once.
static int schedule_twiddles(Plan& p, const KernelInfo* k, const void** dev) {
    std::vector<double> tw;
    int64_t ns = k->rad[0];
    for (int i = 1; i < k->nrad; ++i) {
        const int R = k->rad[i];
        for (int r = 1; r < R; ++r)
            for (int64_t kk = 0; kk < ns; ++kk) {
                double re, im;
                root_of_unity(kk * r, ns * R, &re, &im);
                tw.push_back(re);
                tw.push_back(im);
            }
        ns *= R;
    }
    if (k->prec == 0) {
        std::vector<float> f(tw.begin(), tw.end());
        return upload_table(p, f.data(), f.size() * sizeof(float), dev);
    }
    return upload_table(p, tw.data(), tw.size() * sizeof(double), dev);
}

// Two-level table for W_L^m = hi[m >> sh] * lo[m & (2^sh - 1)].
int split_twiddles(Plan& p, int prec, int64_t L, int* shift, const void** lo, const void** hi) {
    const int sh = (ilog2(L) + 1) / 2;
    const int64_t nlo = 1LL << sh;
    const int64_t nhi = (L + nlo - 1) / nlo;
    std::vector<double> a(2 * nlo), b(2 * nhi);
    for (int64_t i = 0; i < nlo; ++i) root_of_unity(i, L, &a[2 * i], &a[2 * i + 1]);
    for (int64_t i = 0; i < nhi; ++i) root_of_unity(i << sh, L, &b[2 * i], &b[2 * i + 1]);
    *shift = sh;
    int rc;
    if (prec == 0) {
        std::vector<float> fa(a.begin(), a.end()), fb(b.begin(), b.end());
        if ((rc = upload_table(p, fa.data(), fa.size() * 4, lo))) return rc;
        return upload_table(p, fb.data(), fb.size() * 4, hi);
    }
    if ((rc = upload_table(p, a.data(), a.size() * 8, lo))) return rc;
    return upload_table(p, b.data(), b.size() * 8, hi);
}

// Blocks of a column layout in XCD order (xcd_block), given the bytes between
// the rows that a block reads and that it writes.  Neighbouring groups then
// share an L2, which pays wherever their lines overlap; rows a multiple of 8
// KiB apart put all XCDs on the same memory channels instead.  512 MiB batches, plain -> XCD
// order: complex64 512 x 257 1.146 -> 1.100 ms (three axes), 65536 (rows 2 KiB
// apart) 0.384 -> 0.363, 2048 x 512 (4 KiB) 0.497 -> 0.450, 64 x 1000 0.457 ->
// 0.417; 1024 x 1024 (8 KiB) 0.411 -> 0.425, 2^22 (16 KiB) 0.581 -> 0.631, 2^20 (B reads
// rows 16 KiB apart, writes 4 KiB) 0.464 -> 0.508.
static int xcd_order(int64_t in_pitch, int64_t out_pitch) { return in_pitch % 8192 != 0 && out_pitch % 8192 != 0; }

// blocks: of all slices, where the launch may take k's planar form.  Two a CU
// at least: 64 complex128 rows of 8192 points 9.9 -> 10.9 us, 8 images of 512 x
// 512 22.5 -> 23.5, with one block a CU there is nothing to overlap.
static Step make_step(const KernelInfo* k, const KArgs& a, int64_t gx, int64_t gy, const char* what,
                      int64_t blocks = 0) {
    Step s;
    s.fn = k->planar && blocks >= 512 ? k->planar : k->fn;
    s.grid = dim3((unsigned)gx, (unsigned)gy, 1);
    s.block = dim3((unsigned)k->threads, 1, 1);
    s.arg.resize(sizeof(KArgs));
    std::memcpy(s.arg.data(), &a, sizeof(KArgs));
    s.in_field = (int)offsetof(KArgs, in);
    s.out_field = (int)offsetof(KArgs, out);
    s.nt_field = (int)offsetof(KArgs, nt);
    s.name = std::string(what) + "_n" + std::to_string(k->n) + "_e" + std::to_string(k->e) + "_tpb" +
             std::to_string(k->tpb);
    return s;
}

// Launches with more than 65535 slices along y are split; each piece gets its
// own byte offsets.
static void push_sliced(std::vector<Step>& out, Step s, int64_t slices, int64_t in_bd_bytes, int64_t out_bd_bytes) {
    const int64_t maxy = 65535;
    for (int64_t y0 = 0; y0 < slices; y0 += maxy) {
        Step t = s;
        t.grid.y = (unsigned)std::min(maxy, slices - y0);
        t.in_off = s.in_off + y0 * in_bd_bytes;
        t.out_off = s.out_off + y0 * out_bd_bytes;
        out.push_back(t);
    }
}

// One batched 1-D complex transform of length n along a strided axis:
//   element j of transform (y, c) at  y*bd + c*cd + j*nd   (elements)
// c in [0, count), y in [0, slices).  Emits the steps for direction di.
struct AxisJob {
    int64_t n;
    int64_t count;
    int64_t slices;
    int64_t in_cd, in_nd, in_bd;
    int64_t out_cd, out_nd, out_bd;
    int in_role, out_role;
    int64_t in_off, out_off;   // bytes
    double scale;
    int strategy = AFFT_STRATEGY_AUTO;   // forced route (1-D plans)
    int64_t split = 0;                   // forced four-step n1
};

static int emit_axis(Plan& p, int di, const AxisJob& j, std::string& algo);


// MFMA form (AFFT_FLAG_MFMA): complex64 rows of N = 256 .. 16384 (mfma.hip).
const void* mfma_kernel(int n, int var, int dir, int* per_block, int* threads);

// MFMA form of a single-pass row transform (n = 256 .. 16384).
static int emit_mfma(Plan& p, int di, const AxisJob& j, std::string& algo) {
    const int dir = di ? 1 : -1;
    int g = 1, threads = 256;
    const void* fn = mfma_kernel((int)j.n, VAR_ROW, dir, &g, &threads);
    const KernelInfo* k = find_kernel(0, (int)j.n, VAR_ROW, dir);
    if (p.desc.precision != 0 || !fn || !k || j.in_nd != 1 || j.out_nd != 1)
        return set_error(AFFT_ERR_NOT_IMPLEMENTED,
                         "the MFMA form covers complex64 rows of 2^8 .. 2^24 points");
    KArgs a{};
    int rc = schedule_twiddles(p, k, &a.tw);
    if (rc) return rc;
    a.count = j.count;
    a.in_cd = j.in_cd;
    a.out_cd = j.out_cd;
    a.in_nd = a.out_nd = 1;
    a.scale = j.scale;
    Step s;
    s.fn = fn;
    s.grid = dim3((unsigned)((j.count + g - 1) / g), 1, 1);
    s.block = dim3((unsigned)threads, 1, 1);
    s.arg.resize(sizeof(KArgs));
    std::memcpy(s.arg.data(), &a, sizeof(KArgs));
    s.in_field = (int)offsetof(KArgs, in);
    s.out_field = (int)offsetof(KArgs, out);
    s.nt_field = (int)offsetof(KArgs, nt);
    s.in_role = j.in_role;
    s.out_role = j.out_role;
    s.in_off = j.in_off;
    s.out_off = j.out_off;
    s.name = "mfma" + std::to_string(j.n);
    const int es = 8;
    for (int64_t y = 0; y < j.slices; ++y) {
        Step t = s;
        t.in_off += y * j.in_bd * es;
        t.out_off += y * j.out_bd * es;
        p.steps[di].push_back(t);
    }
    if (!algo.empty()) algo += "+";
    algo += "mfma" + std::to_string(j.n) + "r";
    return AFFT_OK;
}

// A strided axis whose columns are contiguous (cd = 1) and too long for 8
// adjacent columns per block: the column loads would fall apart into
// segments of a few bytes.  Four-step on the axis instead, n = n1*n2, both
// passes on many adjacent columns:
//   A: for each (c, k2): FFT over k1 of x[c + (n2*k1 + k2)*S], times
//      W_n^{k2*j1}, into T[(j1*n2 + k2)*count + c]  (blockIdx.y = k2)
//   B: for each (c, j1): FFT over k2 of T, into X[c + (j1 + n1*j2)*S]
static int emit_col_fourstep(Plan& p, int di, const AxisJob& j, std::string& algo) {
    const int prec = p.desc.precision;
    const int dir = di ? 1 : -1;
    const int es = prec ? 16 : 8;
    const int lg = ilog2(j.n);
    const int64_t n1 = 1LL << (lg / 2), n2 = j.n / n1;
    const KernelInfo* ka = find_kernel(prec, (int)n1, VAR_4A, dir);
    const KernelInfo* kb = find_kernel(prec, (int)n2, VAR_COL, dir);
    if (!ka || !kb) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "missing column four-step kernel");
    const size_t need = (size_t)(j.n * j.count * es);
    if (need > p.tmp_bytes[0]) p.tmp_bytes[0] = need;
    int rc;
    KArgs a{};
    if ((rc = schedule_twiddles(p, ka, &a.tw))) return rc;
    if ((rc = split_twiddles(p, prec, j.n, &a.tw4_shift, &a.tw4_lo, &a.tw4_hi))) return rc;
    a.tw4_L = j.n;
    a.tw4_by_y = 1;
    a.count = j.count;
    a.in_cd = 1;
    a.in_nd = n2 * j.in_nd;
    a.in_bd = j.in_nd;
    a.out_cd = 1;
    a.out_nd = n2 * j.count;
    a.out_bd = j.count;
    a.scale = 1.0;
    KArgs b{};
    if ((rc = schedule_twiddles(p, kb, &b.tw))) return rc;
    b.count = j.count;
    b.in_cd = 1;
    b.in_nd = j.count;
    b.in_bd = n2 * j.count;
    b.out_cd = 1;
    b.out_nd = n1 * j.out_nd;
    b.out_bd = j.out_nd;
    b.scale = j.scale;
    a.xcd = xcd_order(a.in_nd * es, a.out_nd * es);
    b.xcd = xcd_order(b.in_nd * es, b.out_nd * es);
    for (int64_t y = 0; y < j.slices; ++y) {
        Step sa = make_step(ka, a, (j.count + ka->tpb - 1) / ka->tpb, n2, "colA");
        sa.in_role = j.in_role;
        sa.in_off = j.in_off + y * j.in_bd * es;
        sa.out_role = ROLE_TMP0;
        sa.out_off = 0;
        p.steps[di].push_back(sa);
        Step sb = make_step(kb, b, (j.count + kb->tpb - 1) / kb->tpb, n1, "colB");
        sb.in_role = ROLE_TMP0;
        sb.in_off = 0;
        sb.out_role = j.out_role;
        sb.out_off = j.out_off + y * j.out_bd * es;
        p.steps[di].push_back(sb);
    }
    if (!algo.empty()) algo += "+";
    algo += "colfourstep" + std::to_string(n1) + "x" + std::to_string(n2);
    return AFFT_OK;
}

static int emit_single(Plan& p, int di, const AxisJob& j, std::string& algo) {
    const int prec = p.desc.precision;
    const int dir = di ? 1 : -1;
    const int es = prec ? 16 : 8;
    if (p.desc.flags & AFFT_FLAG_MFMA) return emit_mfma(p, di, j, algo);
    int var;
    int64_t count = j.count, slices = j.slices;
    int64_t in_cd = j.in_cd, out_cd = j.out_cd, in_bd = j.in_bd, out_bd = j.out_bd;
    if (j.in_nd == 1 && j.out_nd == 1) {
        var = VAR_ROW;
    } else if (j.in_cd == 1 && j.out_cd == 1) {
        var = VAR_COL;
    } else {
        // no unit direction on either axis: one transform per slice
        var = VAR_COL;
        if (count != 1) {
            // fold c into the slice dimension when the slice dimension is trivial
            if (slices != 1) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "layout with no unit stride and two batch axes");
            slices = count;
            in_bd = j.in_cd;
            out_bd = j.out_cd;
            count = 1;
        }
    }
    const KernelInfo* k = find_kernel(prec, (int)j.n, var, dir);
    if (!k) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "no kernel for n=" + std::to_string(j.n));
    // fewer than 8 adjacent columns per block: column loads of under 64 bytes
    if (var == VAR_COL && count >= 16 && k->tpb < 8 && j.n >= 256 && j.in_cd == 1 && j.out_cd == 1 &&
        j.in_nd >= count && j.out_nd >= count)
        return emit_col_fourstep(p, di, j, algo);
    KArgs a{};
    int rc = schedule_twiddles(p, k, &a.tw);
    if (rc) return rc;
    a.count = count;
    a.in_cd = in_cd;
    a.out_cd = out_cd;
    a.in_nd = j.in_nd;
    a.out_nd = j.out_nd;
    a.in_bd = in_bd;
    a.out_bd = out_bd;
    a.scale = j.scale;
    const int64_t gx = (count + k->tpb - 1) / k->tpb;
    // Column groups that start and end on lines share nothing.  There XCD order pays
    // from 64 MiB on; from 8 MiB to there, in what the caches hold, it takes a block
    // away from the XCD whose L2 the pass before has filled (XCD -> plain order: complex128
    // 8 x 32 x 4096 18.5 -> 13.3 us, complex64 64 x 16 x 4096 31.2 -> 28.8, 64 x 64 x 1024 28.1 ->
    // 25.3; the four-step's columns want it at any size: 65536 x 16 13.2 against 15.9).
    const bool lines = j.in_nd * es % 128 == 0 && j.out_nd * es % 128 == 0;
    const int64_t bytes = j.n * count * slices * es;
    a.xcd = var == VAR_COL && xcd_order(j.in_nd * es, j.out_nd * es) &&
            !(lines && bytes >= int64_t(8) << 20 && bytes < int64_t(64) << 20);
    Step s = make_step(k, a, gx, 1, var == VAR_ROW ? "row" : "col", gx * slices);
    // rows whose threads cover less than a line at a time: no streaming, which
    // would take the partial lines to memory one by one (complex64, 512 MiB: 8
    // points 1.62 -> 0.35 ms, 16 3.47 -> 0.45, 128 0.212 -> 0.183)
    if (var == VAR_ROW && (int64_t)(k->n / k->e) * es < 128) s.nt_mask = 0;
    s.in_role = j.in_role;
    s.out_role = j.out_role;
    s.in_off = j.in_off;
    s.out_off = j.out_off;
    push_sliced(p.steps[di], s, slices, in_bd * es, out_bd * es);
    if (!algo.empty()) algo += "+";
    algo += "lds" + std::to_string(j.n) + (var == VAR_ROW ? "r" : "c");
    return AFFT_OK;
}

// Four-step for n = n1*n2 along a unit-stride axis (in_nd == out_nd == 1):
//   A: columns of the n1 x n2 view (stride n2), twiddle W_n^{k1*n2} fused,
//      into tmp at the same positions;
//   B: rows of tmp (length n2), written transposed: X[k1 + n1*k2].
// Intermediate bytes per four-step chunk; AFFT_FOURSTEP_CHUNK_MB overrides
// it (0: the whole batch at once).
static size_t fourstep_chunk_bytes() {
    static const size_t v = [] {
        const char* e = std::getenv("AFFT_FOURSTEP_CHUNK_MB");
        if (!e || !*e) return size_t(128) << 20;
        const long long mb = std::atoll(e);
        return mb > 0 ? size_t(mb) << 20 : ~size_t(0) >> 1;
    }();
    return v;
}

// The four-step split n1 (column length) of a power-of-two length 2^lg: the
// balanced one, except where the gfx950 tuning records show another one
// faster by more than 5 % on average over their shapes of that length:
// complex64 2^20 as 512 x 2048 (7 %), 2^23 as 4096 x 2048 (44 %), 2^24 as
// 8192 x 2048 (7 %); complex128 2^18 as 1024 x 256 (13 %), 2^19 as
// 256 x 2048 (10 %), 2^23 as 4096 x 2048 (32 %).
static int64_t fourstep_split(int prec, int lg) {
    static constexpr int tuned[2][25] = {
        // complex64, by lg
        {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 9, 0, 0, 12, 13},
        // complex128
        {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 10, 8, 0, 0, 0, 12, 0},
    };
    const int t = lg >= 0 && lg < 25 ? tuned[prec ? 1 : 0][lg] : 0;
    return 1LL << (t ? t : lg / 2);
}

static int emit_fourstep(Plan& p, int di, const AxisJob& j, std::string& algo) {
    const int prec = p.desc.precision;
    const int dir = di ? 1 : -1;
    const int es = prec ? 16 : 8;
    if (j.in_nd != 1 || j.out_nd != 1 || !is_pow2(j.n))
        return set_error(AFFT_ERR_NOT_IMPLEMENTED, "four-step needs a unit-stride power-of-two axis");
    const int lg = ilog2(j.n);
    const bool mf = p.desc.flags & AFFT_FLAG_MFMA;
    int64_t n1 = fourstep_split(prec, lg);
    if (mf) {
        // both MFMA passes have lengths in [256, 4096]: the balanced split
        // (n1 <= n2) unless a split is forced
        n1 = j.split ? j.split : (int64_t)1 << (lg / 2);
        if (!is_pow2(n1) || n1 < 256 || n1 > 4096 || j.n / n1 < 256 || j.n / n1 > 4096 || prec != 0)
            return set_error(AFFT_ERR_NOT_IMPLEMENTED,
                             "the MFMA form covers complex64 rows of 2^8 .. 2^24 points");
    } else if (j.split) {
        if (!is_pow2(j.split) || j.split < 2 || j.split >= j.n)
            return set_error(AFFT_ERR_NOT_IMPLEMENTED, "four-step split must be a power of two below n");
        n1 = j.split;
    }
    const int64_t n2 = j.n / n1;
    if (n2 > max_single_pass(prec) || n1 > max_single_pass(prec))
        return set_error(AFFT_ERR_NOT_IMPLEMENTED, "transform too large for this split");
    const KernelInfo* ka = find_kernel(prec, (int)n1, VAR_4A, dir);
    const KernelInfo* kb = find_kernel(prec, (int)n2, VAR_4B, dir);
    if (!ka || !kb) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "missing four-step kernel");
    // per-block transforms and launch shape of the two passes
    int ga = ka->tpb, gb = kb->tpb, ta = ka->threads, tb = kb->threads;
    const void* fa = ka->fn;
    const void* fb = kb->fn;
    if (mf) {
        fa = mfma_kernel((int)n1, VAR_4A, dir, &ga, &ta);
        fb = mfma_kernel((int)n2, VAR_4B, dir, &gb, &tb);
        if (!fa || !fb) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "missing MFMA four-step kernel");
    }
    // Transforms run in chunks of at most fourstep_chunk_bytes() of intermediate
    // data: pass A of a chunk writes TMP0 and pass B reads it back while much
    // of it is still in the 256 MB last-level cache.  Measured on 512 MiB
    // batches: 128 MiB chunks are 0-9 % faster than one pass over the whole
    // batch; 16-64 MiB chunks are slower (too few blocks per launch).
    const int64_t chunk = std::max<int64_t>(1, (int64_t)(fourstep_chunk_bytes() / (size_t)(j.n * es)));
    const int64_t cc = std::min<int64_t>(chunk, j.count);
    const int64_t need = cc * j.n * es;
    if ((size_t)need > p.tmp_bytes[0]) p.tmp_bytes[0] = (size_t)need;
    int rc;
    KArgs a{};
    if ((rc = schedule_twiddles(p, ka, &a.tw))) return rc;
    if ((rc = split_twiddles(p, prec, j.n, &a.tw4_shift, &a.tw4_lo, &a.tw4_hi))) return rc;
    a.tw4_L = j.n;
    a.count = n2;
    a.in_cd = 1;
    a.in_nd = n2;
    a.out_cd = 1;
    a.out_nd = n2;
    a.out_bd = j.n;
    a.scale = 1.0;
    KArgs b{};
    if ((rc = schedule_twiddles(p, kb, &b.tw))) return rc;
    b.count = n1;
    b.in_cd = n2;
    b.in_nd = 1;
    b.in_bd = j.n;
    b.out_cd = 1;
    b.out_nd = n1;
    b.scale = j.scale;
    a.xcd = xcd_order(n2 * es, n2 * es);
    b.xcd = xcd_order(n2 * es, n1 * es);
    // the transforms (c, y): c-major inside each y slice, cc at a time; a
    // launch covers its chunk's c with blockIdx.y
    for (int64_t y = 0; y < j.slices; ++y) {
        for (int64_t c0 = 0; c0 < j.count; c0 += cc) {
            const int64_t cnt = std::min(cc, j.count - c0);
            KArgs aa = a, bb = b;
            aa.in_bd = j.in_cd;
            bb.out_bd = j.out_cd;
            Step sa = make_step(ka, aa, (n2 + ga - 1) / ga, 1, "4stepA");
            sa.fn = fa;
            sa.block = dim3((unsigned)ta, 1, 1);
            sa.in_role = j.in_role;
            sa.in_off = j.in_off + (y * j.in_bd + c0 * j.in_cd) * es;
            sa.out_role = ROLE_TMP0;
            sa.out_off = 0;
            push_sliced(p.steps[di], sa, cnt, j.in_cd * es, j.n * es);
            Step sb = make_step(kb, bb, (n1 + gb - 1) / gb, 1, "4stepB");
            sb.fn = fb;
            sb.block = dim3((unsigned)tb, 1, 1);
            sb.in_role = ROLE_TMP0;
            sb.in_off = 0;
            sb.out_role = j.out_role;
            sb.out_off = j.out_off + (y * j.out_bd + c0 * j.out_cd) * es;
            push_sliced(p.steps[di], sb, cnt, j.n * es, j.out_cd * es);
        }
    }
    if (!algo.empty()) algo += "+";
    algo += (mf ? "mfma_fourstep" : "fourstep") + std::to_string(n1) + "x" + std::to_string(n2);
    return AFFT_OK;
}

// ---- runtime-size mixed radix ------------------------------------------------
const void* mix_kernel(int prec, int var, int dir);
const void* copy_kernel(int prec);

// Radix schedule for a 2/3/5/7-smooth n: radix-16 passes and the
// power-of-two remainder, with the 3s, 5s and 7s first when there are any.
// Empty if n has another prime factor.
std::vector<int> smooth_schedule(int64_t n) {
    std::vector<int> r;
    int64_t m = n;
    int a = 0;
    while (m % 2 == 0) { m /= 2; ++a; }
    std::vector<int> odd;
    for (int q : {3, 5, 7})
        while (m % q == 0) { m /= q; odd.push_back(q); }
    if (m != 1) return {};
    if (odd.empty()) {
        // powers of two: the remainder radix first (the compile-time
        // schedules' order, whose twiddle layout the ragged cores share)
        while (a >= 4) { r.push_back(16); a -= 4; }
        if (a > 0) r.insert(r.begin(), 1 << a);
        return r;
    }
    // Other smooth lengths: odd radices first, then the power-of-two
    // radices.  A radix-R pass writes its outputs R apart while Ns is small;
    // odd strides spread over the LDS banks, strides of 8 or 16 points
    // conflict, so the large power-of-two radices go where Ns is large.
    // Measured on 512 MiB batches: N=6000 0.431 -> 0.386 ms, N=100000
    // 1.044 -> 0.987 ms.
    for (int q : odd) r.push_back(q);
    if (a % 4) r.push_back(1 << (a % 4));
    for (int i = 0; i < a / 4; ++i) r.push_back(16);
    return r;
}

int gen_cap(int prec) { return prec ? 4096 : 8192; }
int gen_row_cap(int prec) { return prec ? 8192 : 16384; }

int64_t next_pow2(int64_t n) {
    int64_t m = 1;
    while (m < n) m <<= 1;
    return m;
}

// Whether one runtime-radix launch holds a transform of n points on this
// layout.
static bool gen_single_fits(int prec, int64_t n, bool rows) {
    return n <= gen_cap(prec) || (rows && n <= gen_row_cap(prec));
}

// Shape of one k_mix launch.
struct MixShape {
    std::vector<int> rad;
    int tpt = 1, g = 1, threads = 64, lds = 0, pitch = 0;
};
// VAR_ROW and Rader's rows; VAR_COL and VAR_4A; VAR_4B; rows of the other kernels that
// do more than one transform (real rows, padded Bluestein, convolution)
enum MixLayout { MIX_ROWS = 0, MIX_COLS = 1, MIX_TROWS = 2, MIX_FUSED = 3 };

// Mean number of LDS bank passes beyond the first of a wave's access to the
// points addr(lane) (< 0: idle lane): the 64 banks of 4 bytes serve 256 bytes
// at a time, 32 complex64 or 16 complex128 points.
template <class Addr>
static double bank_excess(int per, Addr addr) {
    int sum = 0, groups = 0;
    for (int h = 0; h < 64; h += per) {
        int cnt[32] = {0}, mx = 0;
        for (int l = h; l < h + per; ++l) {
            const int64_t x = addr(l);
            if (x >= 0) mx = std::max(mx, ++cnt[x % per]);
        }
        if (mx) { sum += mx; ++groups; }
    }
    return groups ? (double)sum / groups - 1.0 : 0.0;
}

static double mix_bank_excess(const MixShape& m, int64_t n, int prec, MixLayout lay) {
    const int per = prec ? 16 : 32;
    double out = 0;
    int64_t ns = 1;
    for (size_t i = 0; i < m.rad.size(); ++i) {
        const int64_t q = m.rad[i], nr = n / q;
        const bool lanes_c = lay == MIX_COLS || (lay == MIX_TROWS && i + 1 == m.rad.size());
        auto at = [&](int l, bool write) -> int64_t {
            const int64_t c = lanes_c ? l % m.g : l / m.tpt, j = lanes_c ? l / m.g : l % m.tpt;
            if (l >= m.g * m.tpt || j >= nr) return -1;
            const int64_t k = j % ns, x = write ? (j - k) * q + k : j;
            return lay == MIX_COLS ? x * m.g + c : c * m.pitch + x;
        };
        if (i) out += bank_excess(per, [&](int l) { return at(l, false); });
        if (i + 1 < m.rad.size()) out += bank_excess(per, [&](int l) { return at(l, true); });
        ns *= q;
    }
    return out;
}

// Estimated cost of a launch shape, in passes, without the bank conflicts:
// the passes, the lane slots beyond one per point and pass, the resident
// blocks per CU (LDS, and 5 / 3 waves per SIMD), whether there is only one,
// the line segments of the global accesses and the block size.  The
// coefficients are fitted on all schedules, thread counts and group sizes
// of 70 row lengths (24 .. 16128 points), 52 column and 26 transposing cases
// of 512 MiB in both precisions: the pick is on average 2.4 % (rows), 4.4 %
// (columns) and 6.6 % (transposing rows) slower than the best one, 25 % at
// worst.
//
// few: 1 for launches of up to 4 MiB, 0 from 8 MiB on (mix_few); 16 and 32 for Rader's
// rows, which compute longer on as much.  These are over before their blocks have to
// share the CUs: a block's own time decides, the passes and the points that a
// thread takes in turn, little else (of columns not even the conflicts).
// On every shape of 360 row and 184 column
// cases of up to 2^20 points (10 to 8000 a transform, both precisions) the picks are 2.9
// and 3.5 % slower than the best in the mean, 21 and 20 % at worst; by the
// other terms alone 7.7 and 28 %, 62 and 125 % (complex64 columns 625 x 33 11.4 ->
// 5.4 us, 1225 x 500 11.2 -> 8.3).  Columns in several slices and the fused kernels were
// not among them and keep the other terms.
static double mix_few(int64_t n, int64_t count, int64_t slices, int prec, MixLayout lay, bool staged) {
    if (lay == MIX_TROWS || lay == MIX_FUSED || (lay == MIX_COLS && slices > 1)) return 0.0;
    return std::clamp((staged ? 25.0 : 23.0) - std::log2((double)n * count * slices * (prec ? 16 : 8)), 0.0, 1.0);
}

// staged: rows that come through LDS (Rader's): lines and the block size matter less,
// whole waves and conflicts more.  386 cases of 11 to 2017 points, 2^14 to 2^23 in all: 2.7 %
// from the best in the mean, 32 % at worst, by the terms of plain rows 6.0 and 42 %;
// large complex128 launches keep those (4.4 to 7.8 % there, and some lengths 10 to 18 %
// better: 38479 rows of 109 points 27.8 us against 32.9) (441505 complex64 rows of 19 points 57 -> 42 us, 545587 of 13 47 -> 38, 1245 of 421 11.2 -> 8.6).
static double mix_cost(const MixShape& m, int64_t n, int prec, MixLayout lay, int64_t blocks_total, double few,
                       bool staged) {
    const int es = prec ? 16 : 8, wps = prec ? 3 : 5, waves = m.threads / 64;
    const int by_waves = waves <= 8 ? wps * 4 / waves : wps / ((waves + 3) / 4);
    // blocks of exactly half a CU's LDS do not pair: complex128 columns of 640 points, 13107
    // in blocks of 8 (80 KiB) 83 us, of 4 57; of 1280 points 80 and 62
    const int blocks = std::max(1, std::min({(int)(163839 / std::max(m.lds, 1)), by_waves, 32}));
    const double P = (double)m.rad.size(), inv = 1.0 / blocks, one = blocks == 1 ? 1.0 : 0.0, th = m.threads / 1024.0;
    double work = -P, serial = 0;
    for (int q : m.rad) {
        const int64_t rounds = (n / q + m.tpt - 1) / m.tpt;
        work += (double)m.threads / m.g * rounds * q / n;
        serial += (double)rounds * q;
    }
    const double seg = m.g * es, seg128 = std::max(0.0, 128 / seg - 1), seg64 = seg < 64 ? 1.0 : 0.0;
    const double rl = 128.0 / (std::min<int64_t>(m.tpt, n / m.rad.front()) * es);
    const double rs = 128.0 / (std::min<int64_t>(m.tpt, n / m.rad.back()) * es);
    // fewer blocks than CUs: smaller groups spread the work
    const double idle = blocks_total < 256 ? std::log2(256.0 / blocks_total) : 0.0;
    switch (lay) {
    case MIX_ROWS:
    case MIX_FUSED: {
        const double lines = 0.056 * rl + 0.035 * rs + 0.029 * rl * rl + 0.037 * rs * rs;
        const double full = staged && !prec ? 0.2 * work + 0.538 * inv + 0.113 * one + 0.3 * lines - 0.2 * th
                                            : 0.105 * work + 0.538 * inv + 0.113 * one + lines - 0.433 * th;
        return P + few * (1.5 * serial / 64 + 0.1 * th) + (1 - few) * (idle + full);
    }
    case MIX_COLS:
        return P + few * (serial / 64 + 0.4 * th + 0.5 * idle + 0.023 * (seg128 + seg64)) +
               (1 - few) * (idle + 0.546 * work + 1.647 * inv + 3.575 * one + 1.155 * seg128 + 1.173 * seg64 - 1.645 * th);
    default:
        return P + 0.054 * work + 1.81 * inv + 0.05 * one + 0.886 * seg128 + 0.106 * seg64 + 0.205 * rl -
               0.0092 * m.rad.front() - 0.143 * th + idle;
    }
}

static constexpr int kMixRadices[] = {20, 18, 16, 15, 14, 12, 10, 9, 8, 7, 6, 5, 4, 3, 2};

// Fewest passes of a 7-smooth n over kMixRadices (at most `most`).
static int mix_min_passes(int64_t n, int most) {
    if (n == 1) return 0;
    if (most <= 0) return MIX_MAXPASS + 1;
    int best = MIX_MAXPASS + 1;
    for (int q : kMixRadices)
        if (n % q == 0) best = std::min(best, 1 + mix_min_passes(n / q, std::min(most, best - 1) - 1));
    return best;
}

int mix_passes(int64_t n) { return mix_min_passes(n, MIX_MAXPASS); }

// Launch shape of n 7-smooth points: every order of radices with the fewest
// passes, and with one more where they are within a factor 1.7 of each
// other, times every thread count that gives some pass whole butterflies,
// times the group sizes; the bank conflicts rank the cheapest of them.
// Lengths of one pass try any two: from memory such rows are a thread's each, half of them
// a line (2^23 complex64 points in rows of 10, 14 and 18: one pass 46, 47, 54 us, two
// 30 to 33).  Rows with a slot to spare (pad) come through LDS: below 12 points
// one pass is theirs, from 16 on two (16000 complex64 rows of 11 points by Rader's 10
// 5.0 us, 5 x 2 5.6; of 17 by 16 6.3, 4 x 4 5.7; of 19 by 18 7.0, 6 x 3 6.2).
// Radices up to 10 hold 16 points per thread, so at most n/16 threads (the
// largest block at the largest length) always fit.
// pad: LDS slots of a row beyond its n points.
static bool mix_shape(int64_t n, int prec, MixLayout lay, int64_t count, int64_t slices, MixShape& out,
                      double* cost = nullptr, int pad = 0) {
    const int es = prec ? 16 : 8, maxth = prec ? MixCfg<double>::THREADS : MixCfg<float>::THREADS;
    const bool rows = lay == MIX_ROWS || lay == MIX_FUSED;
    const double few = mix_few(n, count, slices, prec, lay, pad > 0);
    const double conf = rows ? 0.02 * few + (pad && !prec ? 0.1 : 0.005) * (1 - few)
                             : (1 - few) * (lay == MIX_COLS ? 0.203 : 0.012);
    const int minp = mix_min_passes(n, MIX_MAXPASS);
    if (minp > MIX_MAXPASS || (lay == MIX_TROWS ? n | 1 : n + pad) * es > 163840) return false;
    // Radices that the largest block holds, and the numbers of passes (bit p:
    // p passes) in which they make up a rest of n: orders that no block size fits
    // are never listed.  (Listing them took up to 15 ms a length; 300 rows of a
    // rough length look at many: plans of 9174 complex64 points 90 -> 2.6 ms, of 10007
    // 41 -> 2.7.)
    auto usable = [&](int q) { return n % q == 0 && (n / q + mix_mb(q) - 1) / mix_mb(q) <= maxth; };
    std::map<int64_t, unsigned> reach{{1, 1u}};
    auto passes_of = [&](auto&& self, int64_t rest) -> unsigned {
        const auto hit = reach.find(rest);
        if (hit != reach.end()) return hit->second;
        unsigned r = 0;
        for (int q : kMixRadices)
            if (rest % q == 0 && usable(q)) r |= self(self, rest / q) << 1;
        return reach[rest] = r;
    };
    std::vector<std::pair<double, MixShape>> top;   // sorted, the cheapest few
    constexpr size_t KEEP = 12;
    std::vector<int> rad;
    auto consider = [&]() {
        int lo = 1;
        for (int q : rad) lo = std::max<int>(lo, (int)((n / q + mix_mb(q) - 1) / mix_mb(q)));
        int tpts[64], nt = 0;
        for (int q : rad)
            for (int m = 1; m <= mix_mb(q); ++m) {
                const int64_t t = (n / q + m - 1) / m;
                if (t < lo || t > maxth) continue;
                bool seen = false;
                for (int i = 0; i < nt; ++i) seen |= tpts[i] == t;
                if (!seen && nt < 64) tpts[nt++] = (int)t;
            }
        for (int i = 0; i < nt; ++i) {
            MixShape m;
            m.tpt = tpts[i];
            int last_g = 0;
            for (int w = 0; w < 6; ++w) {
                if (rows) {
                    static constexpr int want[6] = {64, 128, 192, 256, 512, 0};
                    if (!want[w]) break;
                    m.g = (int)std::min<int64_t>(count, std::max(1, want[w] / m.tpt));
                } else {
                    m.g = 32 >> w;
                }
                if (m.g == last_g) continue;
                last_g = m.g;
                if (m.g > 1 && m.g >= 2 * count) continue;
                m.pitch = (int)(lay == MIX_TROWS ? n | 1 : n + pad);
                const int64_t lds = (int64_t)m.g * m.pitch * es;
                if ((int64_t)m.g * m.tpt > maxth || lds > 163840) continue;
                m.lds = (int)lds;
                m.threads = (m.g * m.tpt + 63) / 64 * 64;
                m.rad = rad;
                const double c = mix_cost(m, n, prec, lay, std::max<int64_t>(1, (count + m.g - 1) / m.g * slices), few, pad > 0);
                if (top.size() == KEEP && c >= top.back().first) continue;
                auto it = top.begin();
                while (it != top.end() && it->first <= c) ++it;
                top.insert(it, {c, m});
                if (top.size() > KEEP) top.pop_back();
            }
        }
    };
    auto extend = [&](auto&& self, int64_t rest, int passes) -> void {
        if (rest == 1) {
            if ((int)rad.size() != passes) return;
            if (passes == minp + 1 && !top.empty()) {
                const auto mm = std::minmax_element(rad.begin(), rad.end());
                if (minp == 1 ? pad && n < 12 : *mm.second * 10 > *mm.first * 17) return;
            }
            consider();
            return;
        }
        const int left = passes - (int)rad.size();
        for (int q : kMixRadices) {
            if (rest % q || !usable(q) || !(passes_of(passes_of, rest / q) >> (left - 1) & 1)) continue;
            rad.push_back(q);
            self(self, rest / q, passes);
            rad.pop_back();
        }
    };
    // more passes only where no schedule of the fewest fits the block size
    for (int passes = pad && n >= 16 ? std::max(2, minp) : minp; passes <= MIX_MAXPASS && (passes <= minp + 1 || top.empty()); ++passes)
        if (passes_of(passes_of, n) >> passes & 1) extend(extend, n, passes);
    if (top.empty()) return false;
    double best = 1e300;
    for (auto& t : top) {
        const double c = t.first + conf * mix_bank_excess(t.second, n, prec, lay);
        if (c < best) {
            best = c;
            out = t.second;
        }
    }
    if (cost) *cost = best;
    return true;
}

std::vector<int> mix_lds_schedule(int64_t n, int prec, int tpt, int pitch) {
    MixShape m, best;
    m.tpt = tpt;
    m.g = std::max(1, 64 / tpt);
    m.pitch = pitch;
    double best_cost = 1e300;
    auto extend = [&](auto&& self, int64_t rest, int passes) -> void {
        if (rest == 1) {
            if ((int)m.rad.size() != passes) return;
            double cost = 0.0;
            for (int q : m.rad) {
                const int64_t rounds = (n / q + tpt - 1) / tpt;
                if (rounds > mix_mb(q)) return;
                cost += (double)tpt * rounds * q / n;
            }
            cost = 0.105 * cost + 0.05 * mix_bank_excess(m, n, prec, MIX_ROWS);
            if (cost < best_cost) {
                best_cost = cost;
                best.rad = m.rad;
            }
            return;
        }
        if ((int)m.rad.size() == passes) return;
        for (int q : kMixRadices) {
            if (rest % q) continue;
            m.rad.push_back(q);
            self(self, rest / q, passes);
            m.rad.pop_back();
        }
    };
    for (int passes = mix_min_passes(n, MIX_MAXPASS); passes <= MIX_MAXPASS && best.rad.empty(); ++passes)
        extend(extend, n, passes);
    return best.rad;
}

MixPass mix_pass_tables(int64_t n, int R, int64_t ns, std::vector<double>& tw) {
    const MixPass ps{R, (int)ns, (int)(n / R), mod_magic((unsigned)ns), (int)(tw.size() / 2)};
    for (int w = 0; ns > 1 && w < mix_ntw(R); ++w)
        for (int64_t k = 0; k < ns; ++k) {
            double re, im;
            root_of_unity(k * mix_twpow(R, w), ns * R, &re, &im);
            tw.push_back(re);
            tw.push_back(im);
        }
    return ps;
}

// Launch shapes and tables of a plan: its two directions and equal axes share
// them.  Creating the plan of 3000-point rows 406 -> 215 us, of 1080 x 1920 real
// images 814 -> 540, of 1200 x 1500 complex128 grids 542 -> 286.
struct MixCache {
    std::map<std::tuple<int64_t, int, int64_t, int64_t, int>, std::pair<MixArgs, MixShape>> known;
    std::map<std::tuple<int64_t, int64_t, int64_t>, BlueRoute> routes;   // by n, count, slices
};

static MixCache& mix_cache(Plan& p) {
    if (!p.mix_cache) p.mix_cache = std::make_shared<MixCache>();
    return *p.mix_cache;
}

// Kernel arguments of a launch shape and their twiddle tables, in a cleared a.
static int mix_args(Plan& p, int64_t n, MixLayout lay, int64_t count, int64_t slices, MixArgs& a, MixShape& m,
                    int pad = 0) {
    MixCache& cache = mix_cache(p);
    const auto key = std::make_tuple(n, (int)lay, count, slices, pad);
    const auto hit = cache.known.find(key);
    if (hit != cache.known.end()) {
        std::tie(a, m) = hit->second;
        return AFFT_OK;
    }
    if (smooth_schedule(n).empty() || !mix_shape(n, p.desc.precision, lay, count, slices, m, nullptr, pad))
        return set_error(AFFT_ERR_NOT_IMPLEMENTED, "no radix schedule");
    a.n = (int)n;
    a.npass = (int)m.rad.size();
    std::vector<double> tw;
    int64_t ns = 1;
    for (int i = 0; i < a.npass; ++i) {
        a.p[i] = mix_pass_tables(n, m.rad[i], ns, tw);
        ns *= m.rad[i];
    }
    a.tpt = m.tpt;
    a.g = m.g;
    a.divm = mod_magic((unsigned)(lay == MIX_COLS ? m.g : m.tpt));
    a.pitch = m.pitch;
    int rc;
    if (p.desc.precision == 0) {
        std::vector<float> f(tw.begin(), tw.end());
        rc = upload_table(p, f.data(), f.size() * 4, &a.k.tw);
    } else {
        rc = upload_table(p, tw.data(), tw.size() * 8, &a.k.tw);
    }
    if (rc == AFFT_OK) cache.known.emplace(key, std::make_pair(a, m));
    return rc;
}

int mix_row_launch(Plan& p, int64_t n, int64_t count, MixArgs& a, int* threads, int* lds) {
    MixShape m;
    const int rc = mix_args(p, n, MIX_FUSED, count, 1, a, m);
    a.k.count = count;
    *threads = m.threads;
    *lds = m.lds;
    return rc;
}

// Non-temporal accesses pay only where a wave covers whole lines: rows whose
// first and last passes run at least 512 contiguous bytes (complex64 60
// points 0.259 -> 0.200 ms without them, 525 0.224 -> 0.204; 960 0.183 ->
// 0.175 with them), columns whose groups start and end on 128-byte lines
// (transposing 400-point rows into rows of 500 0.357 -> 0.251 ms without
// them, into rows of 512 0.196 -> 0.189 with them).
static int mix_nt_mask(const MixShape& m, const MixArgs& a, MixLayout lay, int prec) {
    const int es = prec ? 16 : 8;
    if (lay == MIX_ROWS) {
        const int run = std::min({m.tpt, a.p[0].nr, a.p[a.npass - 1].nr}) * es;
        return run >= 512 ? NT_STORE | NT_LOAD : 0;
    }
    auto lines = [&](long long nd, long long bd) { return (nd * es) % 128 == 0 && (bd * es) % 128 == 0 && (m.g * es) % 128 == 0; };
    int nt = lines(a.k.out_nd, a.k.out_bd) ? NT_STORE : 0;
    if (lay == MIX_COLS && lines(a.k.in_nd, a.k.in_bd)) nt |= NT_LOAD;
    return nt;
}

static Step make_mix_step(const void* fn, const MixArgs& a, const MixShape& m, MixLayout lay, int prec,
                          const std::string& name) {
    Step s;
    s.fn = fn;
    s.grid = dim3((unsigned)((a.k.count + m.g - 1) / m.g), 1, 1);
    s.block = dim3((unsigned)m.threads, 1, 1);
    s.lds_bytes = m.lds;
    s.arg.resize(sizeof(MixArgs));
    std::memcpy(s.arg.data(), &a, sizeof(MixArgs));
    s.in_field = (int)(offsetof(MixArgs, k) + offsetof(KArgs, in));
    s.out_field = (int)(offsetof(MixArgs, k) + offsetof(KArgs, out));
    s.nt_field = (int)(offsetof(MixArgs, k) + offsetof(KArgs, nt));
    s.nt_mask = mix_nt_mask(m, a, lay, prec);
    s.name = name;
    return s;
}

int prep_dynamic_lds(const void* fn, int lds) {
    if (lds > 65536) AFFT_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    return AFFT_OK;
}

static int emit_gen_single(Plan& p, int di, const AxisJob& j, std::string& algo) {
    const int prec = p.desc.precision;
    const int dir = di ? 1 : -1;
    const int es = prec ? 16 : 8;
    if (p.desc.flags & AFFT_FLAG_MFMA) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "mixed radix has no MFMA form");
    int var;
    int64_t count = j.count, slices = j.slices, in_bd = j.in_bd, out_bd = j.out_bd;
    if (j.in_nd == 1 && j.out_nd == 1) var = VAR_ROW;
    else if (j.in_cd == 1 && j.out_cd == 1) var = VAR_COL;
    else {
        var = VAR_COL;
        if (count != 1) {
            if (slices != 1) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "layout with no unit stride and two batch axes");
            slices = count;
            in_bd = j.in_cd;
            out_bd = j.out_cd;
            count = 1;
        }
    }
    if (!gen_single_fits(prec, j.n, var == VAR_ROW))
        return set_error(AFFT_ERR_NOT_IMPLEMENTED, "mixed radix: length too large for one pass on this layout");
    const MixLayout lay = var == VAR_ROW ? MIX_ROWS : MIX_COLS;
    MixArgs g{};
    MixShape m;
    int rc = mix_args(p, j.n, lay, count, slices, g, m);
    if (rc) return rc;
    const void* fn = mix_kernel(prec, var, dir);
    if ((rc = prep_dynamic_lds(fn, m.lds))) return rc;
    g.k.count = count;
    g.k.in_cd = j.in_cd;
    g.k.out_cd = j.out_cd;
    g.k.in_nd = j.in_nd;
    g.k.out_nd = j.out_nd;
    g.k.in_bd = in_bd;
    g.k.out_bd = out_bd;
    g.k.scale = j.scale;
    Step s = make_mix_step(fn, g, m, lay, prec, "mix" + std::to_string(j.n));
    s.in_role = j.in_role;
    s.out_role = j.out_role;
    s.in_off = j.in_off;
    s.out_off = j.out_off;
    push_sliced(p.steps[di], s, slices, in_bd * es, out_bd * es);
    if (!algo.empty()) algo += "+";
    algo += "mixed" + std::to_string(j.n) + (var == VAR_ROW ? "r" : "c");
    return AFFT_OK;
}

// Default split n = n1 x n2 of a smooth four-step: the divisor pair of least
// estimated cost, each factor a power of two held in LDS (the compile-time
// kernel) or a runtime-radix length of 8 to 4096 points (the in-place
// column kernel, at most 16 points per thread), with n1/sqrt(n) in
// [0.2, 5].  A factor costs 3 on the compile-time kernel, else one per pass
// plus one per radix-2 and a half per radix-4 pass (of smooth_schedule's
// radices); ties go to the more balanced pair, then the smaller n1.  Fitted on 33
// complex64 / complex128 lengths from 9000 to 10^6 on kernels with one radix of {2, 3,
// 4, 5, 7, 8, 16} a pass: 5.4 % mean regret there, against 15.6 % for the power-of-two
// part as the column factor.  On the composite radices it is 7.8 % over 599
// shapes of the tuning records, 77 % at worst (12042240 as 735 x 16384 0.237 ms, 3136 x 3840
// 0.134); wisdom and the cost model pick among the timed splits.  Lengths
// with no such pair take the most balanced divisors within the caps.
int64_t gen_fourstep_split(int64_t n, int prec) {
    const int64_t cap = gen_cap(prec), rcap = std::min<int64_t>(cap, 4096);
    auto usable = [&](int64_t m) { return is_pow2(m) ? m <= max_single_pass(prec) : m <= rcap; };
    auto cost = [&](int64_t m) {
        if (is_pow2(m)) return 3.0;
        const std::vector<int> r = smooth_schedule(m);
        double c = (double)r.size();
        for (int q : r) c += q == 2 ? 1.0 : q == 4 ? 0.5 : 0.0;
        return c;
    };
    const double rt = std::sqrt((double)n);
    int64_t n1 = 0;
    double best = 0, bal = 0;
    const int64_t lo = std::max<int64_t>(8, (int64_t)std::ceil(0.2 * rt)), hi = std::min<int64_t>(n / 8, (int64_t)(5.0 * rt));
    for (int64_t d = lo; d <= hi; ++d) {
        if (n % d || !usable(d) || !usable(n / d)) continue;
        const double c = cost(d) + cost(n / d), b = std::fabs(std::log(d / rt));
        if (!n1 || c < best - 1e-9 || (c < best + 1e-9 && b < bal - 1e-9)) {
            n1 = d;
            best = c;
            bal = b;
        }
    }
    if (!n1)
        for (int64_t d = 1; d * d <= n; ++d)
            if (n % d == 0 && d <= cap && n / d <= cap) n1 = d;
    return n1;
}

// Four-step over runtime kernels for smooth n beyond one LDS pass.
static int emit_gen_fourstep(Plan& p, int di, const AxisJob& j, std::string& algo) {
    const int prec = p.desc.precision;
    const int dir = di ? 1 : -1;
    const int es = prec ? 16 : 8;
    if (j.in_nd != 1 || j.out_nd != 1) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "four-step needs unit stride");
    const int cap = gen_cap(prec);
    int64_t n1 = gen_fourstep_split(j.n, prec);
    if (j.split) {
        // a power-of-two factor may use the compile-time kernels' larger cap
        auto fits = [&](int64_t f) { return f <= (is_pow2(f) ? (int64_t)max_single_pass(prec) : (int64_t)cap); };
        if (j.split < 2 || j.n % j.split || !fits(j.split) || !fits(j.n / j.split))
            return set_error(AFFT_ERR_NOT_IMPLEMENTED, "four-step split must divide n into LDS-sized factors");
        n1 = j.split;
    }
    if (!n1) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "no four-step split for n=" + std::to_string(j.n));
    const int64_t n2 = j.n / n1;
    // chunks of transforms whose intermediate data stays in the last-level cache
    const int64_t cc = std::min<int64_t>(j.count, std::max<int64_t>(1, (int64_t)(fourstep_chunk_bytes() / (size_t)(j.n * es))));
    const size_t need = (size_t)(cc * j.n * es);
    if (need > p.tmp_bytes[0]) p.tmp_bytes[0] = need;
    int rc;
    // A power-of-two factor held in LDS runs on the compile-time Stockham
    // kernel of that length, the other factor on the runtime passes.
    const KernelInfo* ka = (is_pow2(n1) && n1 >= 2) ? find_kernel(prec, (int)n1, VAR_4A, dir) : nullptr;
    const KernelInfo* kb = (is_pow2(n2) && n2 >= 2) ? find_kernel(prec, (int)n2, VAR_4B, dir) : nullptr;
    MixArgs ga{}, gb{};
    MixShape ma, mb;
    if (ka) {
        if ((rc = schedule_twiddles(p, ka, &ga.k.tw))) return rc;
    } else if ((rc = mix_args(p, n1, MIX_COLS, n2, cc, ga, ma))) {
        return rc;
    }
    if (kb) {
        if ((rc = schedule_twiddles(p, kb, &gb.k.tw))) return rc;
    } else if ((rc = mix_args(p, n2, MIX_TROWS, n1, cc, gb, mb))) {
        return rc;
    }
    // k_mix reads its four-step tables in double for either precision
    if ((rc = split_twiddles(p, ka ? prec : 1, j.n, &ga.k.tw4_shift, &ga.k.tw4_lo, &ga.k.tw4_hi))) return rc;
    const void* fa = ka ? ka->fn : mix_kernel(prec, VAR_4A, dir);
    const void* fb = kb ? kb->fn : mix_kernel(prec, VAR_4B, dir);
    if ((!ka && (rc = prep_dynamic_lds(fa, ma.lds))) || (!kb && (rc = prep_dynamic_lds(fb, mb.lds)))) return rc;
    ga.k.tw4_L = j.n;
    ga.k.count = n2;
    ga.k.in_cd = 1; ga.k.in_nd = n2; ga.k.out_cd = 1; ga.k.out_nd = n2;
    ga.k.out_bd = j.n;
    ga.k.scale = 1.0;
    gb.k.count = n1;
    gb.k.in_cd = n2; gb.k.in_nd = 1; gb.k.in_bd = j.n;
    gb.k.out_cd = 1; gb.k.out_nd = n1;
    gb.k.scale = j.scale;
    ga.k.xcd = xcd_order(n2 * es, n2 * es);   // read by the compile-time kernels
    gb.k.xcd = xcd_order(n2 * es, n1 * es);
    for (int64_t y = 0; y < j.slices; ++y) {
        for (int64_t c0 = 0; c0 < j.count; c0 += cc) {
            const int64_t cnt = std::min(cc, j.count - c0);
            MixArgs a2 = ga, b2 = gb;
            a2.k.in_bd = j.in_cd;
            b2.k.out_bd = j.out_cd;
            Step sa = ka ? make_step(ka, a2.k, (n2 + ka->tpb - 1) / ka->tpb, 1, "4stepA")
                         : make_mix_step(fa, a2, ma, MIX_COLS, prec, "mix4A");
            sa.in_role = j.in_role;
            sa.in_off = j.in_off + (y * j.in_bd + c0 * j.in_cd) * es;
            sa.out_role = ROLE_TMP0;
            sa.out_off = 0;
            push_sliced(p.steps[di], sa, cnt, j.in_cd * es, j.n * es);
            Step sb = kb ? make_step(kb, b2.k, (n1 + kb->tpb - 1) / kb->tpb, 1, "4stepB")
                         : make_mix_step(fb, b2, mb, MIX_TROWS, prec, "mix4B");
            sb.in_role = ROLE_TMP0;
            sb.in_off = 0;
            sb.out_role = j.out_role;
            sb.out_off = j.out_off + (y * j.out_bd + c0 * j.out_cd) * es;
            push_sliced(p.steps[di], sb, cnt, j.n * es, j.out_cd * es);
        }
    }
    if (!algo.empty()) algo += "+";
    algo += "mixed4step" + std::to_string(n1) + "x" + std::to_string(n2);
    return AFFT_OK;
}

// ---- Bluestein ---------------------------------------------------------------
// In-place iterative radix-2 FFT in long double: builds the Bluestein filter
// spectrum at plan time.
static void host_fft_ld(std::vector<long double>& re, std::vector<long double>& im) {
    const size_t n = re.size();
    for (size_t i = 1, jj = 0; i < n; ++i) {
        size_t bit = n >> 1;
        for (; jj & bit; bit >>= 1) jj ^= bit;
        jj ^= bit;
        if (i < jj) { std::swap(re[i], re[jj]); std::swap(im[i], im[jj]); }
    }
    // twiddles W_n^k, k < n/2, computed once
    std::vector<long double> wr(n / 2 + 1), wi(n / 2 + 1);
    for (size_t k = 0; k < n / 2; ++k) {
        double c, s;
        root_of_unity((int64_t)k, (int64_t)n, &c, &s);
        wr[k] = c;
        wi[k] = s;
    }
    for (size_t len = 2; len <= n; len <<= 1) {
        const size_t half = len / 2, step = n / len;
        for (size_t b = 0; b < n; b += len) {
            for (size_t k = 0; k < half; ++k) {
                const long double cr = wr[k * step], ci = wi[k * step];
                const size_t u = b + k, v = b + k + half;
                const long double xr = re[v] * cr - im[v] * ci, xi = re[v] * ci + im[v] * cr;
                re[v] = re[u] - xr; im[v] = im[u] - xi;
                re[u] += xr; im[u] += xi;
            }
        }
    }
}

// As host_fft_ld for any m (a product of small primes): recursive
// decimation in time by the smallest prime factor.
static void host_dft_ld(const std::complex<long double>* x, int64_t stride, std::complex<long double>* y, int64_t m,
                        const std::complex<long double>* w, int64_t wstep, int64_t total) {
    if (m == 1) {
        y[0] = x[0];
        return;
    }
    int64_t q = 2;
    while (m % q) ++q;
    const int64_t k1 = m / q;
    for (int64_t r = 0; r < q; ++r) host_dft_ld(x + r * stride, stride * q, y + r * k1, k1, w, wstep * q, total);
    std::vector<std::complex<long double>> t(q);
    for (int64_t k = 0; k < k1; ++k) {
        for (int64_t r = 0; r < q; ++r) t[r] = y[r * k1 + k];
        for (int64_t s = 0; s < q; ++s) {
            std::complex<long double> a = t[0];
            for (int64_t r = 1; r < q; ++r) a += t[r] * w[(r * (k + s * k1) % m) * wstep % total];
            y[s * k1 + k] = a;
        }
    }
}

// Forward spectrum of one sequence of m complex128 points, m 7-smooth
// (interleaved re, im in `v`, replaced by its DFT), on the plan's device with a
// complex128 plan of that length, powers of two forced onto their routes
// (never Bluestein).
static int device_fft_c128(Plan& p, std::vector<double>& v, int64_t m) {
    afft_plan_desc d{};
    d.kind = AFFT_C2C;
    d.precision = AFFT_COMPLEX128;
    d.rank = 1;
    d.dims[0] = m;
    d.batch = 1;
    d.strategy = m > (is_pow2(m) ? max_single_pass(1) : gen_row_cap(1)) ? AFFT_STRATEGY_SIXSTEP
                 : is_pow2(m)                                           ? AFFT_STRATEGY_STOCKHAM
                                                                        : AFFT_STRATEGY_MIXED;
    afft_plan sub = nullptr;
    int rc = afft_plan_create_desc(static_cast<afft_context>(p.ctx), &d, &sub);
    if (rc) return rc;
    const size_t bytes = (size_t)m * 16;
    void* buf = nullptr;
    hipError_t e = hipMalloc(&buf, 2 * bytes);
    if (e == hipSuccess) e = hipMemcpy(buf, v.data(), bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        rc = exec_plan(*sub, AFFT_FORWARD, (char*)buf + bytes, buf, sub->stream);
        if (rc == AFFT_OK) e = hipStreamSynchronize(sub->stream);
        if (rc == AFFT_OK && e == hipSuccess) e = hipMemcpy(v.data(), (char*)buf + bytes, bytes, hipMemcpyDeviceToHost);
    }
    if (buf) (void)hipFree(buf);
    afft_plan_destroy(sub);
    if (rc) return rc;
    if (e != hipSuccess) return set_error(AFFT_ERR_DEVICE, std::string("Bluestein filter spectrum: ") + hipGetErrorString(e));
    return AFFT_OK;
}

// The chirp exp(-iπ k²/n) = W_{2n}^{k² mod 2n}, k < n, in FP64.  Above 4096
// points from two long-double tables of about sqrt(2n) roots each,
// W_{2n}^r = W_{2n}^{(r >> s) 2^s} W_{2n}^{r & (2^s - 1)}, multiplied in long
// double and rounded once (the product's error is far below a double ulp).
// AFFT_FLAG_REF_CHIRP uses the reference's unreduced argument π k²/n.
static void bluestein_chirp(int64_t n, bool refchirp, std::vector<double>& ch) {
    ch.assign(2 * n, 0.0);
    if (refchirp) {
        for (int64_t k = 0; k < n; ++k) {
            const double a = -3.14159265358979323846 * (double)(k * k) * (1.0 / (double)n);
            ch[2 * k] = std::cos(a);
            ch[2 * k + 1] = std::sin(a);
        }
        return;
    }
    const int64_t L = 2 * n;
    if (n <= 4096) {
        for (int64_t k = 0, r = 0; k < n; r = (r + 2 * k + 1) % L, ++k)
            root_of_unity(r, L, &ch[2 * k], &ch[2 * k + 1]);   // r = k^2 mod 2n
        return;
    }
    int sh = 0;
    while ((int64_t(1) << (2 * sh)) < L) ++sh;
    const int64_t B = int64_t(1) << sh, H = (L + B - 1) / B;
    std::vector<long double> lr(B), li(B), hr(H), hi(H);
    for (int64_t i = 0; i < B; ++i) root_of_unity_ld(i, L, &lr[i], &li[i]);
    for (int64_t i = 0; i < H; ++i) root_of_unity_ld(i * B, L, &hr[i], &hi[i]);
    for (int64_t k = 0, r = 0; k < n; r = (r + 2 * k + 1) % L, ++k) {
        const int64_t a = r & (B - 1), b = r >> sh;
        ch[2 * k] = (double)(lr[a] * hr[b] - li[a] * hi[b]);
        ch[2 * k + 1] = (double)(lr[a] * hi[b] + li[a] * hr[b]);
    }
}

// A generator of the multiplicative group modulo a prime n.
static int64_t primitive_root(int64_t n) {
    std::vector<int64_t> f;
    for (int64_t r = n - 1, q = 2; r > 1; ++q)
        if (r % q == 0) {
            f.push_back(q);
            while (r % q == 0) r /= q;
        }
    for (int64_t g = 2;; ++g) {
        bool ok = true;
        for (int64_t q : f) {
            int64_t x = 1, b = g;
            for (int64_t e = (n - 1) / q; e; e >>= 1, b = b * b % n)
                if (e & 1) x = x * b % n;
            ok &= x != 1;
        }
        if (ok) return g;
    }
}

static bool is_prime(int64_t n) {
    for (int64_t q = 2; q * q <= n; ++q)
        if (n % q == 0) return false;
    return n > 1;
}

int blue_tables(Plan& p, int64_t n, int64_t m, double inv_scale, BlueTables& bt, int64_t tr_m1) {
    const bool refchirp = p.desc.flags & AFFT_FLAG_REF_CHIRP;
    int rc;
    auto up = [&](const double* v, int64_t len, const void** dev) -> int {
        if (p.desc.precision == 0) {
            std::vector<float> f(v, v + len);
            return upload_table(p, f.data(), f.size() * 4, dev);
        }
        return upload_table(p, v, (size_t)len * 8, dev);
    };
    // chirp and filter spectra are shared by the plan's two directions
    const auto key = std::make_tuple(n, m, tr_m1);
    auto it = p.blue_cache.find(key);
    if (it == p.blue_cache.end()) {
        BlueCache bc;
        std::vector<double> spec(2 * m, 0.0);
        if (tr_m1 == BLUE_RADER) {
            // b[q] = W_n^(g^-q), q < m = n - 1
            std::vector<unsigned short> perm(m);
            const int64_t gen = primitive_root(n);
            for (int64_t q = 0, x = 1; q < m; x = x * gen % n, ++q) {
                perm[q] = (unsigned short)x;
                const int64_t at = q ? m - q : 0;
                root_of_unity(x, n, &spec[2 * at], &spec[2 * at + 1]);
            }
            if ((rc = upload_table(p, perm.data(), perm.size() * 2, &bc.perm))) return rc;
        } else {
            bluestein_chirp(n, refchirp, bc.ch);
        // Forward filter b[k] = conj(chirp[k]), mirrored (b[m-k] = b[k]), zero
        // between.  Its spectrum B: a long-double host FFT up to 4096 points,
        // above that one complex128 FFT on the device (each costs about
        // 0.1-0.5 ms around 4096 points).  The inverse filter is
        // conj(b), whose spectrum is conj(B[-k mod m]).
            spec[0] = bc.ch[0];
            spec[1] = -bc.ch[1];
            for (int64_t k = 1; k < n; ++k) {
                spec[2 * k] = spec[2 * (m - k)] = bc.ch[2 * k];
                spec[2 * k + 1] = spec[2 * (m - k) + 1] = -bc.ch[2 * k + 1];
            }
        }
        if (m <= 4096 && !is_pow2(m)) {
            std::vector<std::complex<long double>> x(m), y(m), w(m);
            for (int64_t k = 0; k < m; ++k) {
                x[k] = {spec[2 * k], spec[2 * k + 1]};
                long double re, im;
                root_of_unity_ld(k, m, &re, &im);
                w[k] = {re, im};
            }
            host_dft_ld(x.data(), 1, y.data(), m, w.data(), 1, m);
            for (int64_t k = 0; k < m; ++k) {
                spec[2 * k] = (double)y[k].real();
                spec[2 * k + 1] = (double)y[k].imag();
            }
        } else if (m <= 4096) {
            std::vector<long double> re(m), im(m);
            for (int64_t k = 0; k < m; ++k) {
                re[k] = spec[2 * k];
                im[k] = spec[2 * k + 1];
            }
            host_fft_ld(re, im);
            for (int64_t k = 0; k < m; ++k) {
                spec[2 * k] = (double)re[k];
                spec[2 * k + 1] = (double)im[k];
            }
        } else if ((rc = device_fft_c128(p, spec, m))) {
            return rc;
        }
        std::unique_ptr<double[]> filt[2];   // not cleared: every entry is written once
        // natural order, or row-major [k1][k2] of k = k1 + tr_m1 * k2
        const int64_t m2 = tr_m1 > 0 ? m / tr_m1 : 0;
        const double dm = (double)m, inv_m = 1.0 / dm;
        const bool exact = is_pow2(m);   // then x * inv_m == x / m, and far cheaper
        auto div = [&](double x) { return exact ? x * inv_m : x / dm; };
        for (int d = 0; d < 2; ++d) filt[d].reset(new double[2 * m]);
        // filt[0][at] = spec[k] / m, filt[1][at] = conj(spec[-k mod m]) / m,
        // through a buffer where the order changes (runs of 32 points read,
        // of 256 points written)
        auto put = [&](const double* f, const double* r, int64_t at) {
            filt[0][2 * at] = div(f[0]);
            filt[0][2 * at + 1] = div(f[1]);
            filt[1][2 * at] = div(r[0]);
            filt[1][2 * at + 1] = div(-r[1]);
        };
        if (tr_m1 > 0) {
            constexpr int64_t T1 = 32, T2 = 256;
            std::vector<double> buf(4 * T1 * (T2 + 1));
            for (int64_t r0 = 0; r0 < tr_m1; r0 += T1) {
                const int64_t n1 = std::min(T1, tr_m1 - r0);
                for (int64_t c0 = 0; c0 < m2; c0 += T2) {
                    const int64_t n2 = std::min(T2, m2 - c0);
                    for (int64_t c = 0; c < n2; ++c)
                        for (int64_t r = 0; r < n1; ++r) {
                            const int64_t k = r0 + r + tr_m1 * (c0 + c), mk_ = (m - k) & (m - 1);   // m is a power of two here
                            double* q = &buf[4 * (r * (T2 + 1) + c)];
                            q[0] = spec[2 * k];
                            q[1] = spec[2 * k + 1];
                            q[2] = spec[2 * mk_];
                            q[3] = spec[2 * mk_ + 1];
                        }
                    for (int64_t r = 0; r < n1; ++r)
                        for (int64_t c = 0; c < n2; ++c) {
                            const double* q = &buf[4 * (r * (T2 + 1) + c)];
                            put(q, q + 2, (r0 + r) * m2 + c0 + c);
                        }
                }
            }
        } else {
            for (int64_t k = 0; k < m; ++k) put(&spec[2 * k], &spec[k ? 2 * (m - k) : 0], k);
        }
        if (tr_m1 != BLUE_RADER && (rc = up(bc.ch.data(), 2 * n, &bc.chirp))) return rc;
        for (int d = 0; d < 2; ++d)
            if ((rc = up(filt[d].get(), 2 * m, &bc.filt[d]))) return rc;
        it = p.blue_cache.emplace(key, std::move(bc)).first;
    }
    const std::vector<double>& ch = it->second.ch;
    bt.chirp = it->second.chirp;
    bt.filt[0] = it->second.filt[0];
    bt.filt[1] = it->second.filt[1];
    bt.perm = it->second.perm;
    if (tr_m1 == BLUE_RADER) return AFFT_OK;
    // post-multiply tables: the chirp itself (forward), conj(chirp) times the
    // inverse scale (inverse)
    bt.post[0] = bt.chirp;
    if (inv_scale == 0.0) return AFFT_OK;
    std::vector<double> post(2 * n);
    for (int64_t k = 0; k < n; ++k) {
        post[2 * k] = ch[2 * k] * inv_scale;
        post[2 * k + 1] = -ch[2 * k + 1] * inv_scale;
    }
    return up(post.data(), 2 * n, &bt.post[1]);
}

static void alias_through_copy(Plan& p, int di, const AxisJob& j);
const void* mix_blue_kernel_c64();
const void* mix_blue_kernel_c128();
const void* mix_rader_kernel_c64();
const void* mix_rader_kernel_c128();

// Rows of a length with a prime factor above 7 on k_mix_blue (kblue.hpp):
// Rader's form (m = n - 1) or Bluestein's with a 7-smooth m >= 2n - 1.
static int emit_mix_blue(Plan& p, int di, const AxisJob& j, int64_t m, bool rader, std::string& algo) {
    const int prec = p.desc.precision;
    const int es = prec ? 16 : 8;
    BlueTables bt;
    MixBlueArgs a{};
    MixShape ms;
    int rc = blue_tables(p, j.n, m, 0.0, bt, rader ? BLUE_RADER : 0);
    if (rc || (rc = mix_args(p, m, rader ? MIX_ROWS : MIX_FUSED, j.count, j.slices, a.m, ms, rader ? 1 : 0))) return rc;
    const void* fn = rader ? (prec ? mix_rader_kernel_c128() : mix_rader_kernel_c64())
                           : (prec ? mix_blue_kernel_c128() : mix_blue_kernel_c64());
    if ((rc = prep_dynamic_lds(fn, ms.lds))) return rc;
    a.chirp = bt.chirp;
    a.filt = bt.filt[di];
    a.perm = (const unsigned short*)bt.perm;
    a.n = (int)j.n;
    a.inverse = di;
    a.m.k.count = j.count;
    a.m.k.in_cd = j.in_cd;
    a.m.k.out_cd = j.out_cd;
    a.m.k.scale = j.scale;
    const std::string name = (rader ? "rader" : "bluestein") + std::to_string(j.n);
    for (int64_t y = 0; y < j.slices; ++y) {
        Step s;
        s.fn = fn;
        s.grid = dim3((unsigned)((j.count + ms.g - 1) / ms.g), 1, 1);
        s.block = dim3((unsigned)ms.threads, 1, 1);
        s.lds_bytes = ms.lds;
        s.arg.resize(sizeof(MixBlueArgs));
        std::memcpy(s.arg.data(), &a, sizeof(MixBlueArgs));
        s.in_field = (int)(offsetof(MixArgs, k) + offsetof(KArgs, in));
        s.out_field = (int)(offsetof(MixArgs, k) + offsetof(KArgs, out));
        s.in_role = j.in_role;
        s.out_role = j.out_role;
        s.in_off = j.in_off + y * j.in_bd * es;
        s.out_off = j.out_off + y * j.out_bd * es;
        s.name = name;
        p.steps[di].push_back(s);
    }
    if (next_pow2(2 * j.n - 1) > max_single_pass(prec)) alias_through_copy(p, di, j);
    if (!algo.empty()) algo += "+";
    algo += name + (rader ? "" : "m" + std::to_string(m));
    return AFFT_OK;
}

// The 7-smooth M >= 2n - 1 that k_mix_blue should take for n, 0 where the power
// of two m does better.  Among the first eight that fit in LDS the least
// modelled time: the launch shape's cost, in which both transforms share the
// trip through memory (0.98 to 1.24 of the best of nine measured at 27 lengths
// from 22 to 9797, mean 1.02).
//
// A point of the compile-time kernel (k_blue) costs less, so M has to be
// shorter by a factor.  2^24 complex64 points, power of two -> M: 131 points 512
// 0.185 ms -> 270 0.109; 341 1024 0.150 -> 686 0.134; 611 2048 0.143 -> 1260
// 0.148; 1111 4096 0.164 -> 2268 0.150; 1313 4096 0.146 -> 2700 0.155; 2053 8192 0.354
// -> 4200 0.191; 6001 16384 0.266 -> 12096 0.215.  2^23 complex128 points: 143 512 0.152
// -> 288 0.114; 703 2048 0.135 -> 1440 0.124; 1529 4096 0.135 -> 3072 0.134; 2587 8192
// 0.217 -> 5184 0.243.  It is also the quicker one through a few rows, up to so
// many points of m: complex64 521, 2048 rows 13.3 against 15.2 us, 8192 44 against
// 42; 2053, 256 rows 13.0 against 13.6, 512 24.6 against 16.1; complex128 521,
// 1024 rows 14.6 against 17.2, 2048 26.4 against 23.2.  Against the three-pass chain always, in up
// to four passes (complex64 8209 points 0.511 -> 0.239 ms, complex128 4099 0.530
// -> 0.233), in more with rows enough: complex64 10007 on 20480 points in six
// passes, 64 rows 0.041 -> 0.046, 256 0.068 -> 0.050.
static int64_t blue_smooth_length(int64_t n, int64_t m, int prec, int64_t count, int64_t slices) {
    double factor = 1.0;
    int64_t fewest = 0;
    if (m < 256) return 0;
    if (m <= max_single_pass(prec)) {
        if (prec) {
            factor = m <= 1024 ? 1.4 : m <= 4096 ? 1.5 : 1.65;
            if (m <= 4096) fewest = 1 << 23;
        } else {
            factor = m <= 1024 ? 1.45 : m <= 4096 ? 1.75 : 1.33;
            fewest = m <= 4096 ? 1 << 24 : m <= 8192 ? 1 << 22 : 0;
        }
    }
    if (count * slices * m < fewest) return 0;
    int64_t best = 0;
    double least = 1e300;
    const int64_t top = std::min<int64_t>((int64_t)((double)m / factor), 163840 / (prec ? 16 : 8));
    for (int64_t c = 2 * n - 1, seen = 0; c <= top && seen < 8; ++c) {
        MixShape ms;
        double cost;
        if (smooth_schedule(c).empty() || !mix_shape(c, prec, MIX_FUSED, count, slices, ms, &cost)) continue;
        ++seen;
        // 256 complex64 points are two passes of the compile-time kernel: 2^23 points of
        // rows of 86 53.7 us, 89.6 padded to 175 = 7 x 5 x 5; of 79 54.3, 55.5 padded to
        // 160 = 10 x 16, whose LDS rows conflict
        if (!prec && m == 256 && (ms.rad.size() > 2 || std::count(ms.rad.begin(), ms.rad.end(), 16))) continue;
        if (m > max_single_pass(prec) && ms.rad.size() > 4 && count * slices < 256) continue;
        if ((cost - 1) * (double)c < least) {
            least = (cost - 1) * (double)c;
            best = c;
        }
    }
    return best;
}

// Plans with the reference's chirp (refchirp) stay on its padded lengths.  Rader's form
// halves the points of the convolution: primes of 2^24 complex64 points, from
// the padded form: 31 points 0.112 -> 0.106 ms, 257 0.215 -> 0.095, 1009 0.138
// -> 0.091, 4051 0.24 -> 0.126, 8101 0.22 -> 0.144; 2^23 complex128: 61 0.115 -> 0.085,
// 1009 0.132 -> 0.092, 8101 0.30 -> 0.175.  A few rows are through the
// compile-time kernel sooner where m is 2048 or 4096 (complex64 1009: 64 rows
// 8.9 against 11.4 us, 1024 11.3 against 11.8, 2048 17.7 against 16.6; 2017: 512
// rows 11.5 against 14.5, 1024 18.2 against 17.6) or very short (17: 64
// rows 5.6 against 5.7).
// Where the power of two is beyond LDS a row is one block's, the chain spreads
// it over many: one launch from 64 rows on (complex128 4099 points, chain -> one
// launch: 1 row 19.5 -> 25.7 us, 32 27.5 -> 26.3, 64 31.3 -> 26.7, 256 67 -> 33;
// complex64 18433: 1 row 19.9 -> 41.5, 64 43.4 -> 42.8, 256 122 -> 52).
BlueRoute blue_route(int64_t n, int prec, int64_t count, int64_t slices, bool refchirp, bool rader) {
    const int64_t m = next_pow2(2 * n - 1);
    if (!refchirp && (m <= max_single_pass(prec) || count * slices >= 64)) {
        MixShape ms;
        const int64_t fewest = m <= 128 ? 1 << 15 : m <= 1024 || m > 4096 ? 0 : 1 << 22;
        if (rader && count * slices * m >= fewest && n < 65536 && is_prime(n) && !smooth_schedule(n - 1).empty() &&
            mix_shape(n - 1, prec, MIX_ROWS, count, slices, ms, nullptr, 1))
            return {BLUE_ROUTE_RADER, n - 1, 1};
        if (const int64_t sm = blue_smooth_length(n, m, prec, count, slices)) return {BLUE_ROUTE_SMOOTH, sm, 1};
    }
    return {BLUE_ROUTE_POW2, m, m <= max_single_pass(prec) ? 1 : 3};
}

static int emit_bluestein(Plan& p, int di, const AxisJob& j, std::string& algo) {
    const int prec = p.desc.precision;
    const int dir = di ? 1 : -1;
    const int es = prec ? 16 : 8;
    if (j.in_nd != 1 || j.out_nd != 1) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "Bluestein needs unit stride");
    const int64_t n = j.n, m = next_pow2(2 * n - 1);
    auto& routes = mix_cache(p).routes;
    const auto key = std::make_tuple(n, j.count, j.slices);
    if (!routes.count(key))
        routes[key] = blue_route(n, prec, j.count, j.slices, p.desc.flags & AFFT_FLAG_REF_CHIRP,
                                 p.desc.strategy != AFFT_STRATEGY_BLUESTEIN);
    const BlueRoute route = routes[key];
    if (route.kind != BLUE_ROUTE_POW2) return emit_mix_blue(p, di, j, route.m, route.kind == BLUE_ROUTE_RADER, algo);
    if (m <= max_single_pass(prec)) {
        BlueTables bt;
        int rc = blue_tables(p, n, m, 0.0, bt);
        if (rc) return rc;
        const KernelInfo* k = find_kernel(prec, (int)m, VAR_BLUE, dir);
        if (!k) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "no Bluestein kernel for M=" + std::to_string(m));
        KArgs dummy{};
        int rc2 = schedule_twiddles(p, k, &dummy.tw);
        if (rc2) return rc2;
        BArgs b{};
        b.tw = dummy.tw;
        b.chirp = bt.chirp;
        b.filt = bt.filt[di];
        b.count = j.count;
        b.in_cd = j.in_cd;
        b.out_cd = j.out_cd;
        b.nlog = n;
        b.scale = j.scale;
        Step s;
        s.fn = k->fn;
        s.grid = dim3((unsigned)((j.count + k->tpb - 1) / k->tpb), 1, 1);
        s.block = dim3((unsigned)k->threads, 1, 1);
        s.arg.resize(sizeof(BArgs));
        std::memcpy(s.arg.data(), &b, sizeof(BArgs));
        s.in_field = (int)offsetof(BArgs, in);
        s.out_field = (int)offsetof(BArgs, out);
        s.in_role = j.in_role;
        s.out_role = j.out_role;
        s.in_off = j.in_off;
        s.out_off = j.out_off;
        s.name = "bluestein" + std::to_string(n);
        for (int64_t y = 0; y < j.slices; ++y) {
            Step t = s;
            t.in_off += y * j.in_bd * es;
            t.out_off += y * j.out_bd * es;
            p.steps[di].push_back(t);
        }
        if (!algo.empty()) algo += "+";
        algo += "bluestein" + std::to_string(n) + "m" + std::to_string(m);
        return AFFT_OK;
    }
    // chained form of M = m1*m2: column pass (chirp and zero padding fused
    // into its loads), row pass (k_bluemid: forward FFT, filter, inverse FFT),
    // inverse column pass (post-chirp and crop fused into its stores), all in
    // place in TMP0
    const int lg = ilog2(m);
    // Rows of 4096 points where that leaves columns of 128 to 1024 points.
    // Complex128 1,000,003 points x 8 (M = 2^21) with m1 = 128, 256, 512, 1024:
    // 0.403, 0.384, 0.384, 0.390 ms; complex64 40,009 x 256 (M = 2^17) with 128,
    // 256, 512: 0.272, 0.310, 0.296.
    int64_t m1 = std::max<int64_t>(128, m / 4096);
    if (m1 > 1024) m1 = 1LL << (lg / 2);
    const int64_t m2 = m / m1;
    if (m2 > max_single_pass(prec)) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "Bluestein length too large");
    const KernelInfo* ka = find_kernel(prec, (int)m1, VAR_4A, -1);
    const KernelInfo* kr = find_kernel(prec, (int)m2, VAR_BLUEMID, -1);
    const KernelInfo* kc = find_kernel(prec, (int)m1, VAR_COL, 1);
    if (!ka || !kr || !kc) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "missing Bluestein chain kernel");
    BlueTables bt;
    // the inverse scale rides on the post-multiply table
    int rc = blue_tables(p, n, m, di ? j.scale : 0.0, bt, m1);
    if (rc) return rc;
    // chunks of transforms whose M-point intermediate stays in the last-level
    // cache between the three passes
    const int64_t cc = std::min<int64_t>(j.count, std::max<int64_t>(1, (int64_t)(fourstep_chunk_bytes() / (size_t)(m * es))));
    const size_t need = (size_t)(cc * m * es);
    if (need > p.tmp_bytes[0]) p.tmp_bytes[0] = need;
    KArgs A{}, R{}, C{};
    if ((rc = schedule_twiddles(p, ka, &A.tw))) return rc;
    if ((rc = split_twiddles(p, prec, m, &A.tw4_shift, &A.tw4_lo, &A.tw4_hi))) return rc;
    A.tw4_L = m;
    A.count = m2;
    A.in_cd = 1; A.in_nd = m2; A.in_bd = j.in_cd;
    A.out_cd = 1; A.out_nd = m2; A.out_bd = m;
    A.scale = 1.0;
    A.xcd = xcd_order(m2 * es, m2 * es);
    A.fuse = FUSE_CHIRP_IN;
    A.fvec = bt.chirp;
    A.fconj = di;
    A.flen = n;
    if ((rc = schedule_twiddles(p, kr, &R.tw))) return rc;
    R.tw4_shift = A.tw4_shift; R.tw4_lo = A.tw4_lo; R.tw4_hi = A.tw4_hi; R.tw4_L = m;
    R.count = m1;
    R.in_cd = R.out_cd = m2; R.in_nd = R.out_nd = 1; R.in_bd = R.out_bd = m;
    R.scale = 1.0;
    R.fvec = bt.filt[di];
    if ((rc = schedule_twiddles(p, kc, &C.tw))) return rc;
    C.count = m2;
    C.in_cd = C.out_cd = 1; C.in_nd = C.out_nd = m2; C.in_bd = m; C.out_bd = j.out_cd;
    C.scale = di ? 1.0 : j.scale;   // normalised and unitary forward plans
    C.xcd = A.xcd;
    C.fuse = FUSE_CROP_OUT;
    C.fvec = bt.post[di];
    C.flen = n;
    for (int64_t y = 0; y < j.slices; ++y) {
        for (int64_t c0 = 0; c0 < j.count; c0 += cc) {
            const int64_t cnt = std::min(cc, j.count - c0);
            Step s1 = make_step(ka, A, (m2 + ka->tpb - 1) / ka->tpb, 1, "blueA");
            s1.in_role = j.in_role; s1.in_off = j.in_off + (y * j.in_bd + c0 * j.in_cd) * es;
            s1.out_role = ROLE_TMP0; s1.out_off = 0;
            push_sliced(p.steps[di], s1, cnt, j.in_cd * es, m * es);
            Step s2 = make_step(kr, R, (m1 + kr->tpb - 1) / kr->tpb, 1, "blueR");
            s2.in_role = s2.out_role = ROLE_TMP0; s2.in_off = s2.out_off = 0;
            push_sliced(p.steps[di], s2, cnt, m * es, m * es);
            Step s3 = make_step(kc, C, (m2 + kc->tpb - 1) / kc->tpb, 1, "blueC", (m2 + kc->tpb - 1) / kc->tpb * cnt);
            s3.in_role = ROLE_TMP0; s3.in_off = 0;
            s3.out_role = j.out_role; s3.out_off = j.out_off + (y * j.out_bd + c0 * j.out_cd) * es;
            push_sliced(p.steps[di], s3, cnt, m * es, j.out_cd * es);
        }
    }
    if (!algo.empty()) algo += "+";
    algo += "bluestein" + std::to_string(n) + "m" + std::to_string(m1) + "x" + std::to_string(m2);
    return AFFT_OK;
}

// ---- copies (length-1 axes, gathers) ------------------------------------------
static Step make_copy(int prec, int64_t lines, int64_t len, int64_t icd, int64_t ind, int64_t ocd, int64_t ond,
                      double scale) {
    CopyArgs c{};
    c.lines = lines;
    c.len = len;
    c.in_cd = icd; c.in_nd = ind; c.out_cd = ocd; c.out_nd = ond;
    c.scale = scale;
    Step s;
    s.fn = copy_kernel(prec);
    const int64_t tot = lines * len;
    s.grid = dim3((unsigned)((tot + 255) / 256), 1, 1);
    s.block = dim3(256, 1, 1);
    s.arg.resize(sizeof(CopyArgs));
    std::memcpy(s.arg.data(), &c, sizeof(CopyArgs));
    s.in_field = (int)offsetof(CopyArgs, in);
    s.out_field = (int)offsetof(CopyArgs, out);
    s.name = "copy";
    return s;
}

static int emit_axis_direct(Plan& p, int di, const AxisJob& j, std::string& algo);

// The last step is one launch from the caller's input to its output where
// other lengths take several through scratch.  Where src and dst overlap and
// are not the same rows, it reads a packed copy instead (alias_steps): blocks
// would overwrite what others have yet to read.
static void alias_through_copy(Plan& p, int di, const AxisJob& j) {
    if (p.desc.rank != 1 || j.slices != 1 || j.in_role != ROLE_SRC || j.out_role != ROLE_DST) return;
    const bool rows = j.in_nd == 1;
    Step c = make_copy(p.desc.precision, j.count, j.n, j.in_cd, j.in_nd, rows ? j.n : 1, rows ? 1 : j.count, 1.0);
    c.in_role = ROLE_SRC;
    c.in_off = j.in_off;
    c.out_role = ROLE_WORK2;
    Step s = p.steps[di].back();
    KArgs k;   // first in every argument block of k_mix's kernels
    std::memcpy(&k, s.arg.data(), sizeof(k));
    k.in_cd = rows ? j.n : 1;
    k.in_nd = rows ? 1 : j.count;
    std::memcpy(s.arg.data(), &k, sizeof(k));
    s.in_role = ROLE_WORK2;
    s.in_off = 0;
    p.alias_steps[di] = {c, s};
    p.alias_from[di] = p.steps[di].size();
    p.alias_same_ok[di] = j.in_cd == j.out_cd && j.in_nd == j.out_nd;
    p.alias_bytes[di] = (size_t)(j.count * j.n) * (p.desc.precision ? 16 : 8);
}
static_assert(offsetof(MixArgs, k) == 0 && offsetof(MixBlueArgs, m) == 0, "KArgs first");

// Paths that need unit-stride rows get strided lines through a gather into
// TMP1, the row transform in place there, and a scatter back.
static int emit_via_gather(Plan& p, int di, const AxisJob& j, std::string& algo) {
    const int prec = p.desc.precision;
    const int es = prec ? 16 : 8;
    const int64_t lines = j.count * j.slices;
    const size_t need = (size_t)(lines * j.n * es);
    if (need > p.tmp_bytes[1]) p.tmp_bytes[1] = need;
    for (int64_t y = 0; y < j.slices; ++y) {
        Step g = make_copy(prec, j.count, j.n, j.in_cd, j.in_nd, j.n, 1, 1.0);
        g.in_role = j.in_role; g.in_off = j.in_off + y * j.in_bd * es;
        g.out_role = ROLE_TMP1; g.out_off = y * j.count * j.n * es;
        p.steps[di].push_back(g);
    }
    AxisJob r = j;
    r.count = lines;
    r.slices = 1;
    r.in_cd = r.out_cd = j.n;
    r.in_nd = r.out_nd = 1;
    r.in_bd = r.out_bd = 0;
    r.in_role = r.out_role = ROLE_TMP1;
    r.in_off = r.out_off = 0;
    int rc = emit_axis_direct(p, di, r, algo);
    if (rc) return rc;
    for (int64_t y = 0; y < j.slices; ++y) {
        Step s = make_copy(prec, j.count, j.n, j.n, 1, j.out_cd, j.out_nd, 1.0);
        s.in_role = ROLE_TMP1; s.in_off = y * j.count * j.n * es;
        s.out_role = j.out_role; s.out_off = j.out_off + y * j.out_bd * es;
        p.steps[di].push_back(s);
    }
    algo += "(gathered)";
    return AFFT_OK;
}

static bool needs_rows(const Plan& p, int64_t n, int strategy) {
    const int prec = p.desc.precision;
    if (strategy == AFFT_STRATEGY_SIXSTEP || strategy == AFFT_STRATEGY_BLUESTEIN) return true;
    if ((n & (n - 1)) == 0) return n > max_single_pass(prec);
    if (!smooth_schedule(n).empty()) return n > gen_cap(prec);
    return true;  // Bluestein
}

static int emit_axis_direct(Plan& p, int di, const AxisJob& j, std::string& algo) {
    const int prec = p.desc.precision;
    const bool smooth = !smooth_schedule(j.n).empty();
    const bool rows = j.in_nd == 1 && j.out_nd == 1;
    if ((p.desc.flags & AFFT_FLAG_MFMA) &&
        (!is_pow2(j.n) || j.strategy == AFFT_STRATEGY_MIXED || j.strategy == AFFT_STRATEGY_BLUESTEIN))
        return set_error(AFFT_ERR_NOT_IMPLEMENTED,
                         "the MFMA form covers powers of two on the Stockham and four-step routes only");
    switch (j.strategy) {
    case AFFT_STRATEGY_AUTO: break;
    case AFFT_STRATEGY_STOCKHAM:
        if (is_pow2(j.n) && j.n <= max_single_pass(prec)) return emit_single(p, di, j, algo);
        return set_error(AFFT_ERR_NOT_IMPLEMENTED, "Stockham strategy needs a power of two held in LDS");
    case AFFT_STRATEGY_MIXED:
        if (smooth && gen_single_fits(prec, j.n, rows)) return emit_gen_single(p, di, j, algo);
        return set_error(AFFT_ERR_NOT_IMPLEMENTED, "mixed-radix strategy needs a 7-smooth size held in LDS");
    case AFFT_STRATEGY_SIXSTEP:
        if (is_pow2(j.n)) return emit_fourstep(p, di, j, algo);
        if (smooth) return emit_gen_fourstep(p, di, j, algo);
        return set_error(AFFT_ERR_NOT_IMPLEMENTED, "four-step strategy needs a 7-smooth size");
    case AFFT_STRATEGY_BLUESTEIN:
        if (j.n >= 2) return emit_bluestein(p, di, j, algo);
        return set_error(AFFT_ERR_NOT_IMPLEMENTED, "Bluestein needs n >= 2");
    default:
        return set_error(AFFT_ERR_NOT_IMPLEMENTED, "unknown strategy");
    }
    // Rows of 16 points up to 512 bytes: the compile-time kernel gives a row 2
    // to 8 threads, whose stores are partial lines; the runtime-radix kernel's
    // go line by line.  512 MiB batches, both without streaming stores:
    // complex64 16 points 0.449 -> 0.209 ms, 32 0.237 -> 0.206, 64 0.203 ->
    // 0.184; complex128 16 0.304 -> 0.177, 32 0.198 -> 0.172.  8 points and
    // fewer are one thread's either way (complex64 8 points 0.350 against
    // 0.388), and at 1 KiB the compile-time kernel wins on cached batches
    // (complex64 128 points, 32 MiB: 11.7 against 14.2 us).
    // Rows of 64 complex64 points before other axes stay there beyond 16 MiB, where the
    // next pass finds more of its input in its L2 (32 MiB: 16 x 64 x 4096 29.0 -> 25.5 us,
    // 64 x 64 x 1024 25.3 -> 24.3, 64 x 64 x 64 x 16 37.7 -> 34.9; 8 MiB and 128 MiB even).
    const bool inner64 = p.desc.rank > 1 && !prec && j.n == 64 && j.count * j.slices > 32768;
    if (is_pow2(j.n) && rows && j.n >= 16 && j.n * (prec ? 16 : 8) <= 512 && !inner64 &&
        !(p.desc.flags & AFFT_FLAG_MFMA))
        return emit_gen_single(p, di, j, algo);
    // Long power-of-two columns, many side by side: 32 KiB of column and more
    // leave the compile-time kernel fewer than 8 in a block, hence its two-pass
    // form (emit_col_fourstep); the runtime-radix kernel holds 4 of 32 KiB in one
    // pass.  Two passes -> one: complex128 2048 points, 256 columns 17.4 -> 11.4 us,
    // 2048 51 -> 34, 4096 88 -> 64, 10000 258 -> 189; 4096 points, 1000 columns 51 -> 38;
    // complex64 4096 points, 256 columns 17.6 -> 13.3, 4096 86 -> 77, 10000 269 -> 224.
    // Not from 256 MiB on where the pitch is a multiple of 8 KiB: complex64 4096 x
    // 8192 222 -> 280.
    if (is_pow2(j.n) && j.in_cd == 1 && j.out_cd == 1 && j.in_nd >= j.count && j.out_nd >= j.count && j.count >= 128 &&
        j.n * (prec ? 16 : 8) >= 32768 && gen_single_fits(prec, j.n, false) && !(p.desc.flags & AFFT_FLAG_MFMA)) {
        const int64_t es = prec ? 16 : 8, pitch = std::max(j.in_nd, j.out_nd) * es;
        if (xcd_order(j.in_nd * es, j.out_nd * es) || pitch * j.n < (int64_t(256) << 20)) {
            const int rc = emit_gen_single(p, di, j, algo);
            if (rc == AFFT_OK) alias_through_copy(p, di, j);
            return rc;
        }
    }
    if (is_pow2(j.n) && j.n <= max_single_pass(prec)) return emit_single(p, di, j, algo);
    if (is_pow2(j.n)) return emit_fourstep(p, di, j, algo);
    if (!smooth_schedule(j.n).empty()) {
        if (gen_single_fits(prec, j.n, rows)) return emit_gen_single(p, di, j, algo);
        return emit_gen_fourstep(p, di, j, algo);
    }
    return emit_bluestein(p, di, j, algo);
}

static int emit_axis(Plan& p, int di, const AxisJob& j, std::string& algo) {
    const int prec = p.desc.precision;
    const int es = prec ? 16 : 8;
    if (j.n == 1) {
        for (int64_t y = 0; y < j.slices; ++y) {
            Step s = make_copy(prec, j.count, 1, j.in_cd, 1, j.out_cd, 1, j.scale);
            s.in_role = j.in_role; s.in_off = j.in_off + y * j.in_bd * es;
            s.out_role = j.out_role; s.out_off = j.out_off + y * j.out_bd * es;
            p.steps[di].push_back(s);
        }
        if (!algo.empty()) algo += "+";
        algo += "copy";
        return AFFT_OK;
    }
    if (needs_rows(p, j.n, j.strategy) && (j.in_nd != 1 || j.out_nd != 1)) return emit_via_gather(p, di, j, algo);
    return emit_axis_direct(p, di, j, algo);
}

// Complex transforms over the axes `axes` (processed in the given order) of
// a row-major array with dims cd[0..rank-1]; batch copies at distances
// in_dist / out_dist (elements).  The first axis reads `in_role`, every axis
// writes `out_role`, later axes work in place there.
static int emit_nd_axes(Plan& p, int di, int rank, const int64_t* cd, const std::vector<int>& axes, int64_t batch,
                        int in_role, int64_t in_dist, int out_role, int64_t out_dist, std::string& algo) {
    int64_t total = 1;
    for (int i = 0; i < rank; ++i) total *= cd[i];
    bool first = true;
    for (int ax : axes) {
        const int64_t len = cd[ax];
        int64_t inner = 1;
        for (int i = ax + 1; i < rank; ++i) inner *= cd[i];
        const int64_t outer = total / (len * inner);
        if (len == 1 && !(first && in_role != out_role)) continue;   // identity axis
        AxisJob j{};
        j.n = len;
        j.scale = di ? 1.0 / (double)len : 1.0;
        j.in_role = first ? in_role : out_role;
        j.out_role = out_role;
        const int64_t idd = first ? in_dist : out_dist;
        if (inner == 1) {
            if (idd == total && out_dist == total) {
                j.count = outer * batch; j.slices = 1;
                j.in_cd = len; j.in_nd = 1; j.in_bd = 0;
                j.out_cd = len; j.out_nd = 1; j.out_bd = 0;
            } else {
                j.count = outer; j.slices = batch;
                j.in_cd = len; j.in_nd = 1; j.in_bd = idd;
                j.out_cd = len; j.out_nd = 1; j.out_bd = out_dist;
            }
            int rc = emit_axis(p, di, j, algo);
            if (rc) return rc;
        } else {
            // columns: count = inner adjacent columns, slices = outer (per batch
            // copy, or across all copies when they are packed)
            const int es = p.desc.precision ? 16 : 8;
            const bool packed = idd == total && out_dist == total;
            const int64_t nb = packed ? 1 : batch;
            for (int64_t b = 0; b < nb; ++b) {
                AxisJob k = j;
                k.count = inner;
                k.slices = packed ? outer * batch : outer;
                k.in_cd = 1; k.in_nd = inner; k.in_bd = len * inner;
                k.out_cd = 1; k.out_nd = inner; k.out_bd = len * inner;
                k.in_off = b * idd * es;
                k.out_off = b * out_dist * es;
                int rc = emit_axis(p, di, k, algo);
                if (rc) return rc;
            }
        }
        first = false;
    }
    return AFFT_OK;
}

const void* rpost_kernel(int prec, int dir);
const void* mix_real_kernel(int prec, int dir);

// Real rows of n reals (h = n/2 complex points): `rows` rows, row r of slice y
// at y*bd + r*rd (complex elements of each side; the real side counts the
// row as h complex).  R2C when di == 0, C2R when di == 1.
static int emit_real_rows(Plan& p, int di, int64_t n, int64_t rows, int64_t slices, int in_role, int64_t in_rd,
                          int64_t in_bd, int out_role, int64_t out_rd, int64_t out_bd, double scale,
                          std::string& algo) {
    const int prec = p.desc.precision;
    const int es = prec ? 16 : 8;
    const int dir = di ? 1 : -1;
    const int64_t h = n / 2;
    // W_N^k, k < h
    std::vector<double> w(2 * (h + 1));
    for (int64_t k = 0; k <= h; ++k) root_of_unity(k, n, &w[2 * k], &w[2 * k + 1]);
    const void* wk;
    int rc;
    if (prec == 0) {
        std::vector<float> f(w.begin(), w.end());
        rc = upload_table(p, f.data(), f.size() * 4, &wk);
    } else {
        rc = upload_table(p, w.data(), w.size() * 8, &wk);
    }
    if (rc) return rc;
    // Rows of 32 and 64 reals: as the complex ones, too few threads a row in the
    // compile-time kernel.  256 MiB of reals, compile-time -> runtime-radix
    // kernel, R2C / C2R: float32 32 points 0.196 / 0.179 -> 0.153 / 0.131 ms, 64 0.180 /
    // 0.148 -> 0.150 / 0.137; float64 32 0.175 / 0.212 -> 0.120 / 0.118.  128 points
    // are mixed (R2C 0.140 -> 0.121, C2R 0.117 -> 0.133), 16 lose (0.158 -> 0.232).  Under
    // 1024 rows the compile-time kernel is quicker through (64 float32 points, 1 row
    // 4.2 against 4.9 us).
    const bool shortr = (h == 16 || h == 32) && rows * slices >= 1024;
    const KernelInfo* k = (h >= 2 && is_pow2(h) && !shortr) ? find_kernel(prec, (int)h, VAR_REAL, dir) : nullptr;
    if (k) {
        RArgs a{};
        KArgs tmpk{};
        if ((rc = schedule_twiddles(p, k, &tmpk.tw))) return rc;
        a.tw = tmpk.tw;
        a.wk = wk;
        a.count = rows;
        a.in_d = in_rd;
        a.out_d = out_rd;
        a.scale = di ? scale / (double)h : scale;
        for (int64_t y = 0; y < slices; ++y) {
            Step s;
            s.fn = k->fn;
            s.grid = dim3((unsigned)((rows + k->tpb - 1) / k->tpb), 1, 1);
            s.block = dim3((unsigned)k->threads, 1, 1);
            s.arg.resize(sizeof(RArgs));
            std::memcpy(s.arg.data(), &a, sizeof(RArgs));
            s.in_field = (int)offsetof(RArgs, in);
            s.out_field = (int)offsetof(RArgs, out);
            s.in_role = in_role;
            s.out_role = out_role;
            s.in_off = y * in_bd * es;
            s.out_off = y * out_bd * es;
            s.name = di ? "c2r" : "r2c";
            p.steps[di].push_back(s);
        }
        if (!algo.empty()) algo += "+";
        algo += (di ? "c2r" : "r2c") + std::to_string(n);
        return AFFT_OK;
    }
    // smooth h held in LDS: the runtime-radix kernel with the recombination
    if (h >= 2 && (!is_pow2(h) || shortr) && !smooth_schedule(h).empty() && h <= gen_row_cap(prec)) {
        MixRealArgs a{};
        MixShape m;
        if ((rc = mix_args(p, h, MIX_FUSED, rows, slices, a.m, m))) return rc;
        const void* fn = mix_real_kernel(prec, dir);
        if ((rc = prep_dynamic_lds(fn, m.lds))) return rc;
        a.wk = wk;
        a.m.k.count = rows;
        a.m.k.in_cd = in_rd;
        a.m.k.out_cd = out_rd;
        a.m.k.scale = di ? scale / (double)h : scale;
        for (int64_t y = 0; y < slices; ++y) {
            Step s;
            s.fn = fn;
            s.grid = dim3((unsigned)((rows + m.g - 1) / m.g), 1, 1);
            s.block = dim3((unsigned)m.threads, 1, 1);
            s.lds_bytes = m.lds;
            s.arg.resize(sizeof(MixRealArgs));
            std::memcpy(s.arg.data(), &a, sizeof(MixRealArgs));
            s.in_field = (int)(offsetof(MixArgs, k) + offsetof(KArgs, in));
            s.out_field = (int)(offsetof(MixArgs, k) + offsetof(KArgs, out));
            s.in_role = in_role;
            s.out_role = out_role;
            s.in_off = y * in_bd * es;
            s.out_off = y * out_bd * es;
            s.name = di ? "mixc2r" : "mixr2c";
            p.steps[di].push_back(s);
        }
        if (in_role == ROLE_SRC && out_role == ROLE_DST) {
            // the same rows from a packed copy in WORK2, as large as the
            // buffer of the two-launch form
            const int64_t row = di ? h + 1 : h;
            p.alias_same_ok[di] = in_rd == out_rd && (slices == 1 || in_bd == out_bd);
            p.alias_bytes[di] = (size_t)(slices * rows * row * es);
            std::vector<Step>& al = p.alias_steps[di];
            const int64_t copies = rows == 1 ? 1 : slices;
            for (int64_t y = 0; y < copies; ++y) {
                Step cp = rows == 1 ? make_copy(prec, slices, row, in_bd, 1, row, 1, 1.0)
                                    : make_copy(prec, rows, row, in_rd, 1, row, 1, 1.0);
                cp.in_role = ROLE_SRC;
                cp.in_off = y * in_bd * es;
                cp.out_role = ROLE_WORK2;
                cp.out_off = y * rows * row * es;
                al.push_back(cp);
            }
            a.m.k.in_cd = row;
            const size_t first = p.steps[di].size() - (size_t)slices;
            for (int64_t y = 0; y < slices; ++y) {
                Step s = p.steps[di][first + y];
                std::memcpy(s.arg.data(), &a, sizeof(MixRealArgs));
                s.in_role = ROLE_WORK2;
                s.in_off = y * rows * row * es;
                al.push_back(s);
            }
            p.alias_from[di] = p.steps[di].size();
        }
        if (!algo.empty()) algo += "+";
        algo += (di ? "c2r" : "r2c") + std::to_string(n);
        return AFFT_OK;
    }
    // unfused: h-point complex transform as its own steps plus a recombination
    const size_t need = (size_t)(slices * rows * (h + 1) * es);
    if (need > p.tmp_bytes[ROLE_WORK2 - 2]) p.tmp_bytes[ROLE_WORK2 - 2] = need;
    auto post = [&](int irole, int64_t ird, int64_t ibd, int orole, int64_t ord, int64_t obd, double sc) {
        RPArgs r{};
        r.wk = wk;
        r.rows = rows;
        r.h = h;
        r.in_d = ird;
        r.out_d = ord;
        r.scale = sc;
        const int64_t per = di ? h : h + 1;
        for (int64_t y = 0; y < slices; ++y) {
            Step s;
            s.fn = rpost_kernel(prec, dir);
            s.grid = dim3((unsigned)((rows * per + 255) / 256), 1, 1);
            s.block = dim3(256, 1, 1);
            s.arg.resize(sizeof(RPArgs));
            std::memcpy(s.arg.data(), &r, sizeof(RPArgs));
            s.in_field = (int)offsetof(RPArgs, in);
            s.out_field = (int)offsetof(RPArgs, out);
            s.in_role = irole;
            s.out_role = orole;
            s.in_off = y * ibd * es;
            s.out_off = y * obd * es;
            s.name = "rpost";
            p.steps[di].push_back(s);
        }
    };
    AxisJob j{};
    j.n = h;
    j.count = rows;
    j.slices = slices;
    j.in_nd = j.out_nd = 1;
    if (!di) {
        j.in_role = in_role; j.in_cd = in_rd; j.in_bd = in_bd;
        j.out_role = ROLE_WORK2; j.out_cd = h; j.out_bd = rows * h;
        j.scale = 1.0;
        if ((rc = emit_axis(p, di, j, algo))) return rc;
        post(ROLE_WORK2, h, rows * h, out_role, out_rd, out_bd, scale);
    } else {
        post(in_role, in_rd, in_bd, ROLE_WORK2, h, rows * h, 1.0);
        j.in_role = ROLE_WORK2; j.in_cd = h; j.in_bd = rows * h;
        j.out_role = out_role; j.out_cd = out_rd; j.out_bd = out_bd;
        j.scale = scale / (double)h;
        if ((rc = emit_axis(p, di, j, algo))) return rc;
    }
    algo += di ? "(c2r)" : "(r2c)";
    return AFFT_OK;
}

// Planner's choice for AFFT_STRATEGY_AUTO on a 1-D axis: wisdom for this
// size first, then the context's cost model, else the built-in routing
// (cf. planner.go:43-78: registry, wisdom, heuristic).
// MFMA plans keep the MFMA routing: wisdom and the cost model rank the
// plain kernels, and their picks (mixed radix, Bluestein, other four-step
// splits) have no MFMA form.
uint64_t wisdom_features(const Context& c, const afft_plan_desc& d);   // tune.cpp

void choose_strategy(Plan& p, AxisJob& j) {
    if (j.in_nd != 1 || j.out_nd != 1) return;
    if (p.desc.flags & AFFT_FLAG_MFMA) return;
    Context* c = p.ctx;
    std::lock_guard<std::mutex> lock(c->mu);
    auto it = c->wisdom.find(std::make_tuple(j.n, p.desc.precision, wisdom_features(*c, p.desc)));
    Candidate pick{0, 0};
    if (it != c->wisdom.end()) {
        if (parse_strategy(it->second.algorithm, &pick)) {
            j.strategy = pick.strategy;
            j.split = pick.split;
        }
        return;
    }
    if (!c->model) return;
    std::vector<Candidate> cand = plan_candidates(p.desc);
    if (cand.size() < 2) return;
    std::vector<float> x(cand.size() * NFEAT), y(cand.size());
    for (size_t i = 0; i < cand.size(); ++i) plan_features(p.desc, cand[i], &x[i * NFEAT]);
    if (mlp_predict_host(c->model, x.data(), (int64_t)cand.size(), y.data()) != AFFT_OK) return;
    size_t best = 0;
    for (size_t i = 1; i < cand.size(); ++i)
        if (y[i] < y[best]) best = i;
    j.strategy = cand[best].strategy;
    j.split = cand[best].split;
}

static int build_plan_steps(Plan& p) {
    afft_plan_desc& d = p.desc;
    if (d.precision != AFFT_COMPLEX64 && d.precision != AFFT_COMPLEX128)
        return set_error(AFFT_ERR_NOT_IMPLEMENTED, "unknown precision");
    if (d.rank < 1 || d.rank > 8) return set_error(AFFT_ERR_INVALID_LENGTH, "rank must be 1..8");
    int64_t n = 1;
    for (int i = 0; i < d.rank; ++i) {
        if (d.dims[i] < 1) return set_error(AFFT_ERR_INVALID_LENGTH, "dimension must be >= 1");
        n *= d.dims[i];
    }
    if (d.batch == 0) d.batch = 1;
    if (d.batch < 1) return set_error(AFFT_ERR_INVALID_LENGTH, "batch must be >= 1");
    if (d.istride < 0 || d.ostride < 0 || d.idist < 0 || d.odist < 0)
        return set_error(AFFT_ERR_INVALID_STRIDE, "negative stride or distance");
    p.n = n;
    const int es = d.precision ? 16 : 8;
    const int rs = es / 2;
    const bool real = d.kind == AFFT_R2C || d.kind == AFFT_C2R;
    if (!real && d.kind != AFFT_C2C) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "unknown transform kind");
    double fscale = 1.0;
    if (d.flags & AFFT_FLAG_NORMALIZE) fscale = 1.0 / (double)n;
    if (d.flags & AFFT_FLAG_UNITARY) fscale = 1.0 / std::sqrt((double)n);

    if (!real) {
        const int64_t is = d.istride ? d.istride : 1, os = d.ostride ? d.ostride : 1;
        const int64_t id = d.idist ? d.idist : n * is, od = d.odist ? d.odist : n * os;
        if (d.rank > 1 && (is != 1 || os != 1))
            return set_error(AFFT_ERR_INVALID_STRIDE, "N-D plans take unit element stride");
        p.in_elems[0] = p.in_elems[1] = (d.batch - 1) * id + (n - 1) * is + 1;
        p.out_elems[0] = p.out_elems[1] = (d.batch - 1) * od + (n - 1) * os + 1;
        p.in_esize[0] = p.in_esize[1] = p.out_esize[0] = p.out_esize[1] = es;
        for (int di = 0; di < 2; ++di) {
            std::string algo;
            if (d.rank == 1) {
                AxisJob j{};
                j.n = n;
                j.scale = di ? 1.0 / (double)n : fscale;
                j.in_role = ROLE_SRC;
                j.out_role = ROLE_DST;
                j.count = d.batch;
                j.slices = 1;
                j.in_cd = id; j.in_nd = is;
                j.out_cd = od; j.out_nd = os;
                j.strategy = d.strategy;
                j.split = d.split;
                if (!j.strategy) choose_strategy(p, j);
                int rc = emit_axis(p, di, j, algo);
                if (rc) return rc;
            } else {
                std::vector<int> axes;
                for (int ax = d.rank - 1; ax >= 0; --ax) axes.push_back(ax);
                if (n == 1) axes = {d.rank - 1};
                int rc = emit_nd_axes(p, di, d.rank, d.dims, axes, d.batch, ROLE_SRC, id, ROLE_DST, od, algo);
                if (rc) return rc;
                if (p.steps[di].empty()) {
                    // all axes of length 1 but src != dst: plain copy
                    AxisJob j{};
                    j.n = 1; j.count = d.batch * n; j.slices = 1;
                    j.in_cd = 1; j.out_cd = 1; j.in_nd = j.out_nd = 1;
                    j.in_role = ROLE_SRC; j.out_role = ROLE_DST; j.scale = 1.0;
                    if ((rc = emit_axis(p, di, j, algo))) return rc;
                }
                if (!di && fscale != 1.0) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "normalised N-D forward");
            }
            if (di == 0) p.algo = "hip_" + algo;
        }
        return AFFT_OK;
    }

    // ---- real transforms (PlanRealT, PlanReal2D/3D) --------------------------
    const int64_t w = d.dims[d.rank - 1];
    if (w < 2 || (w & 1)) return set_error(AFFT_ERR_INVALID_LENGTH, "real transforms need an even last dimension");
    if ((d.istride && d.istride != 1) || (d.ostride && d.ostride != 1))
        return set_error(AFFT_ERR_INVALID_STRIDE, "real transforms take unit element stride");
    const int64_t h = w / 2, hw = h + 1;
    const int64_t outer = n / w;
    int64_t cd[8];
    for (int i = 0; i < d.rank; ++i) cd[i] = d.dims[i];
    cd[d.rank - 1] = hw;
    const int64_t creal = n, ccx = outer * hw;
    const int64_t rdist = d.idist ? d.idist : creal;   // real side, reals
    const int64_t cdist = d.odist ? d.odist : ccx;     // complex side, complex elements
    if (rdist & 1) return set_error(AFFT_ERR_INVALID_STRIDE, "real-side batch distance must be even");
    // [0] forward: reals in, complex out; [1] inverse: complex in, reals out
    p.in_elems[0] = (d.batch - 1) * rdist + creal;
    p.out_elems[0] = (d.batch - 1) * cdist + ccx;
    p.in_elems[1] = p.out_elems[0];
    p.out_elems[1] = p.in_elems[0];
    p.in_esize[0] = p.out_esize[1] = rs;
    p.out_esize[0] = p.in_esize[1] = es;
    const int64_t rd2 = rdist / 2;   // real batch distance in complex units
    for (int di = 0; di < 2; ++di) {
        std::string algo;
        std::vector<int> axes;
        for (int ax = d.rank - 2; ax >= 0; --ax) axes.push_back(ax);
        int rc;
        // rows are contiguous within one batch copy: outer rows of h / hw
        const bool flat = (rdist == creal && cdist == ccx);
        const int64_t rows = flat ? outer * d.batch : outer;
        const int64_t slices = flat ? 1 : d.batch;
        if (!di) {
            rc = emit_real_rows(p, 0, w, rows, slices, ROLE_SRC, h, rd2, ROLE_DST, hw, cdist, fscale, algo);
            if (rc) return rc;
            if (!axes.empty()) {
                if (fscale != 1.0) return set_error(AFFT_ERR_NOT_IMPLEMENTED, "normalised N-D real forward");
                rc = emit_nd_axes(p, 0, d.rank, cd, axes, d.batch, ROLE_DST, cdist, ROLE_DST, cdist, algo);
                if (rc) return rc;
            }
            p.algo = "hip_" + algo;
        } else {
            int src_role = ROLE_SRC;
            int64_t src_dist = cdist;
            if (!axes.empty()) {
                // outer axes first (inverse order of the forward), into WORK
                std::vector<int> inv_axes(axes.rbegin(), axes.rend());
                const size_t need = (size_t)(d.batch * ccx * es);
                if (need > p.tmp_bytes[ROLE_WORK - 2]) p.tmp_bytes[ROLE_WORK - 2] = need;
                rc = emit_nd_axes(p, 1, d.rank, cd, inv_axes, d.batch, ROLE_SRC, cdist, ROLE_WORK, ccx, algo);
                if (rc) return rc;
                src_role = ROLE_WORK;
                src_dist = ccx;
            }
            const bool flat2 = (rdist == creal && src_dist == ccx);
            const int64_t rows2 = flat2 ? outer * d.batch : outer;
            const int64_t slices2 = flat2 ? 1 : d.batch;
            rc = emit_real_rows(p, 1, w, rows2, slices2, src_role, hw, src_dist, ROLE_DST, h, rd2, 1.0, algo);
            if (rc) return rc;
        }
    }
    return AFFT_OK;
}

Launches launches_for(Plan& p, int di, const void* dst, const void* src) {
    const char* s0 = (const char*)src;
    const char* d0 = (const char*)dst;
    const bool apart = s0 + (size_t)p.in_elems[di] * p.in_esize[di] <= d0 ||
                       d0 + (size_t)p.out_elems[di] * p.out_esize[di] <= s0;
    const bool own = p.alias_steps[di].empty() || apart || (src == dst && p.alias_same_ok[di]);
    Launches l{own ? p.steps[di] : p.alias_steps[di], {}};
    std::copy(p.tmp_bytes, p.tmp_bytes + NTMP, l.bytes);
    if (!own) l.bytes[ROLE_WORK2 - 2] = std::max(l.bytes[ROLE_WORK2 - 2], p.alias_bytes[di]);
    return l;
}

size_t buffer_bytes(const Plan& p, int t) {
    return t == ROLE_WORK2 - 2 ? std::max({p.tmp_bytes[t], p.alias_bytes[0], p.alias_bytes[1]}) : p.tmp_bytes[t];
}

// Rows whose other route takes its scratch in chunks (fourstep_chunk_bytes):
// a longer copy is allocated by the first call that needs it.  The other
// routes of real rows and of columns hold the whole batch.
constexpr size_t kRowAliasReserve = size_t(128) << 20;

int reserve_alias(Plan& p, hipStream_t s) {
    constexpr int t = ROLE_WORK2 - 2;
    if (p.alias_reserved || p.tmp[t] || buffer_bytes(p, t) == p.tmp_bytes[t]) return AFFT_OK;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    AFFT_HIP(hipStreamIsCapturing(s, &cs));
    if (cs != hipStreamCaptureStatusNone) return AFFT_OK;
    p.alias_reserved = true;
    if (p.desc.kind == AFFT_C2C && p.desc.istride <= 1 && buffer_bytes(p, t) > kRowAliasReserve) return AFFT_OK;
    // without the memory only calls over their input fail, when they ask for it
    if (hipMalloc(&p.tmp[t], buffer_bytes(p, t)) != hipSuccess) {
        (void)hipGetLastError();
        p.tmp[t] = nullptr;
    }
    return AFFT_OK;
}

// Enqueues steps on s, with the roles resolved to src, dst and the workspace
// buffers tmp[0 .. NTMP).
int launch_steps(std::vector<Step>& steps, void* dst, const void* src, void* const* tmp, hipStream_t s) {
    void* base[ROLE_COUNT] = {const_cast<void*>(src), dst, tmp[0], tmp[1], tmp[2], tmp[3]};
    for (Step& st : steps) {
        char* ip = (char*)base[st.in_role] + st.in_off;
        char* op = (char*)base[st.out_role] + st.out_off;
        std::memcpy(st.arg.data() + st.in_field, &ip, sizeof(void*));
        std::memcpy(st.arg.data() + st.out_field, &op, sizeof(void*));
        void* args[] = {st.arg.data()};
        AFFT_HIP(hipLaunchKernel(st.fn, st.grid, st.block, args, (size_t)st.lds_bytes, s));
    }
    return AFFT_OK;
}

// A plan's workspace (tmp[]) is shared by all its executions.  When one
// execution is enqueued on a different stream than the previous one, the new
// stream first waits for the previous use to finish, so a plan may be driven
// from several streams (and host threads) without racing on its scratch.
// Under stream capture the caller orders the graph's nodes and no event is
// touched.
int exec_plan(Plan& p, int dir, void* dst, const void* src, hipStream_t s) {
    const int di = dir == AFFT_INVERSE ? 1 : 0;
    const Launches l = launches_for(p, di, dst, src);
    bool ws = false;
    for (int t = 0; t < NTMP; ++t) {
        if (!l.bytes[t]) continue;
        ws = true;
        if (!p.tmp[t]) AFFT_HIP(hipMalloc(&p.tmp[t], buffer_bytes(p, t)));
    }
    if (ws) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        AFFT_HIP(hipStreamIsCapturing(s, &cs));
        if (cs != hipStreamCaptureStatusNone) {
            ws = false;
        } else {
            if (!p.ws_done) AFFT_HIP(hipEventCreateWithFlags(&p.ws_done, hipEventDisableTiming));
            if (p.ws_used && p.ws_stream != s) AFFT_HIP(hipStreamWaitEvent(s, p.ws_done, 0));
        }
    }
    int rc = launch_steps(l.steps, dst, src, p.tmp, s);
    if (rc) return rc;
    if (ws) {
        AFFT_HIP(hipEventRecord(p.ws_done, s));
        p.ws_stream = s;
        p.ws_used = true;
    }
    return AFFT_OK;
}

// Launches that write the caller's output store it non-temporally when that
// output is at least kStreamOutBytes: larger outputs would be evicted from the
// last-level cache before anyone re-reads them, and bypassing it measured
// about 2 % faster on the 512 MiB batches.  A launch that also reads the
// caller's input of that size streams its loads as well (one pass from
// source to destination): about 3 % more on the N=4096 batch, while
// streaming loads alone lose.
constexpr size_t kStreamOutBytes = size_t(128) << 20;

// The steps behind the fused real rows are the same for overlapping buffers.
static void finish_alias_steps(Plan& p) {
    for (int di = 0; di < 2; ++di)
        if (!p.alias_steps[di].empty())
            p.alias_steps[di].insert(p.alias_steps[di].end(), p.steps[di].begin() + p.alias_from[di], p.steps[di].end());
}

int build_plan(Plan& p) {
    int rc = build_plan_steps(p);
    if (rc) return rc;
    finish_alias_steps(p);
    for (int di = 0; di < 2; ++di) {
        const size_t ob = (size_t)p.out_elems[di] * p.out_esize[di];
        const size_t ib = (size_t)p.in_elems[di] * p.in_esize[di];
        if (ob < kStreamOutBytes) continue;
        for (Step& st : p.steps[di]) {
            if (st.out_role != ROLE_DST || st.nt_field < 0) continue;
            int flags = NT_STORE;
            if (st.in_role == ROLE_SRC && ib >= kStreamOutBytes) flags |= NT_LOAD;
            flags &= st.nt_mask;
            std::memcpy(st.arg.data() + st.nt_field, &flags, sizeof(int));
        }
    }
    return AFFT_OK;
}

}  // namespace afft
