"""The composite-radix runtime kernel (kmix.hpp) where its launch shapes have
edges: every radix alone, groups that leave a partial block, several
butterflies a thread, prime-power and longest lengths, in place, strided
columns, four-step factors of a single pass, real rows, and the three-pass
Bluestein chain; against the oracle (numpy for the last), within
the library's budgets (helpers.c64_tol, C128_TOL)."""
import numpy as np
import pytest
import torch

import algofft_hip as A
from algofft_hip import synth
import pyoracle as O
from helpers import C128_TOL, c64_tol, rel_l2

pytestmark = pytest.mark.gpu

PRECS = [(A.COMPLEX64, np.complex64), (A.COMPLEX128, np.complex128)]


def _tol(prec, n):
    return c64_tol(n) if prec == A.COMPLEX64 else C128_TOL


# one pass (3 .. 20), two and three passes, powers of one prime, the longest
# rows of either precision
ROWS = [3, 5, 6, 7, 9, 10, 12, 14, 15, 18, 20, 21, 24, 28, 54, 175, 360, 525, 686, 2187, 2401, 3125, 7938, 8100]


@pytest.mark.parametrize("prec,dt", PRECS)
@pytest.mark.parametrize("n", ROWS + [14406, 15625, 16200, 16384 - 256])
def test_rows_with_partial_groups(ctx, n, prec, dt):
    if prec == A.COMPLEX128 and n > 8192:
        pytest.skip("longer complex128 rows take the four-step route")
    batch = 67 if n < 1000 else 3
    x = synth.uniform_complex(7 * n, (batch, n), dt)
    with A.Plan.from_desc(ctx, (n,), precision=prec, batch=batch) as p:
        assert p.describe() == f"hip_mixed{n}r"
        got = np.empty_like(x)
        p.forward(got, x)
        back = got.copy()
        p.inverse(back, back)   # in place
    assert rel_l2(got, O.fft_batch(x.astype(np.complex128))) <= _tol(prec, n)
    assert rel_l2(back, O.fft_batch(got.astype(np.complex128), inverse=True)) <= _tol(prec, n)


@pytest.mark.parametrize("prec,dt", PRECS)
@pytest.mark.parametrize("n,cols", [(6, 1), (20, 5), (175, 33), (360, 17), (1200, 7), (2401, 3), (4000, 2)])
def test_strided_columns_with_partial_groups(ctx, n, cols, prec, dt):
    # columns of a matrix wider than the batch: element stride cols + 2
    w = cols + 2
    buf = synth.uniform_complex(n + cols, (n, w), dt)
    with A.Plan.from_desc(ctx, (n,), precision=prec, batch=cols, istride=w, idist=1, ostride=w, odist=1) as p:
        out = np.zeros_like(buf)
        p.forward(out.ravel(), buf.ravel())
    ref = O.fft_batch(np.ascontiguousarray(buf[:, :cols].T).astype(np.complex128)).T
    assert rel_l2(out[:, :cols], ref) <= _tol(prec, n)


@pytest.mark.parametrize("prec,dt", PRECS)
@pytest.mark.parametrize("n,split", [(18 * 15, 18), (20 * 20, 20), (12 * 343, 343), (9 * 175, 9), (4050, 2025)])
def test_fourstep_single_pass_factors(ctx, n, split, prec, dt):
    x = synth.uniform_complex(3 * n, (3, n), dt)
    with A.Plan.from_desc(ctx, (n,), precision=prec, batch=3, strategy=A.STRATEGY_SIXSTEP, split=split) as p:
        assert p.describe() == f"hip_mixed4step{split}x{n // split}"
        got = np.empty_like(x)
        p.forward(got, x)
    assert rel_l2(got, O.fft_batch(x.astype(np.complex128))) <= _tol(prec, n)


REAL_H = [3, 5, 9, 12, 18, 20, 21, 50, 175, 525, 960, 2401, 5400, 7938]


@pytest.mark.parametrize("prec", [A.COMPLEX64, A.COMPLEX128])
@pytest.mark.parametrize("h", REAL_H + [16200])
def test_real_rows(ctx, h, prec):
    if prec == A.COMPLEX128 and h > 8192:
        pytest.skip("longer complex128 rows run unfused")
    rdt = np.float32 if prec == A.COMPLEX64 else np.float64
    cdt = np.complex64 if prec == A.COMPLEX64 else np.complex128
    n, batch = 2 * h, 67 if h < 1000 else 3
    x = synth.uniform_real(h, (batch, n), rdt)
    with A.Plan.from_desc(ctx, (n,), precision=prec, kind=A.R2C, batch=batch) as p:
        X = np.empty((batch, h + 1), cdt)
        p.forward(X, x)
        y = np.empty_like(x)
        p.inverse(y, X)
    assert rel_l2(X, O.rfft(x.astype(np.float64))) <= _tol(prec, n)
    assert rel_l2(y, O.irfft(X.astype(np.complex128), n)) <= _tol(prec, n)


@pytest.mark.parametrize("dims", [(50,), (1050,), (6, 50)])
@pytest.mark.parametrize("noalloc", [False, True])
def test_real_rows_over_their_own_input(ctx, dims, noalloc):
    """Packed real plans with dst at src: a row's output lies over the next
    row's input, so the input is copied first."""
    batch, n = 37, dims[-1]
    rows = batch * int(np.prod(dims[:-1], dtype=np.int64))
    x = synth.uniform_real(n, (batch,) + dims, np.float32)
    X = np.fft.rfftn(x.astype(np.float64), axes=tuple(range(1, len(dims) + 1)))
    buf = torch.zeros(rows * (n // 2 + 1) * 2, dtype=torch.float32, device="cuda")
    s = torch.cuda.Stream()
    import ctypes
    fn = A.lib().afft_plan_exec_device_noalloc if noalloc else A.lib().afft_plan_exec_device
    with A.Plan.from_desc(ctx, dims, kind=A.R2C, batch=batch) as p:
        buf[:x.size] = torch.from_numpy(x.ravel()).cuda()
        torch.cuda.synchronize()
        for d in (A.FORWARD, A.INVERSE):
            A.check(fn(p.h, d, ctypes.c_void_p(buf.data_ptr()), ctypes.c_void_p(buf.data_ptr()),
                       ctypes.c_void_p(s.cuda_stream)))
            s.synchronize()
            if d == A.FORWARD:
                got = torch.view_as_complex(buf.view(-1, 2)).cpu().numpy().reshape(X.shape)
                assert rel_l2(got, X) <= c64_tol(x[0].size)
    assert rel_l2(buf[:x.size].cpu().numpy().reshape(x.shape), x) <= 2 * c64_tol(x[0].size)


# three-pass Bluestein chains: padded lengths from the first beyond LDS, rows of
# 128 to 4096 points, both directions
@pytest.mark.parametrize("prec,dt", PRECS)
@pytest.mark.parametrize("n", [4099, 8209, 11 * 1009, 17 * 1031, 70001, 150001, 300007])
def test_bluestein_chain(ctx, n, prec, dt):
    batch = max(1, min(3, 400000 // n))
    x = synth.uniform_complex(n, (batch, n), dt)
    with A.Plan.from_desc(ctx, (n,), precision=prec, batch=batch) as p:
        got = np.empty_like(x)
        p.forward(got, x)
        back = got.copy()
        p.inverse(back, back)
    assert rel_l2(got, np.fft.fft(x.astype(np.complex128), axis=1)) <= _tol(prec, n)
    assert rel_l2(back, np.fft.ifft(got.astype(np.complex128), axis=1)) <= _tol(prec, n)


@pytest.mark.parametrize("prec,dt", PRECS)
@pytest.mark.parametrize("n", [2, 4, 8, 16, 32, 64, 128])
@pytest.mark.parametrize("batch", [1, 67, 4099])
def test_short_power_of_two_rows(ctx, n, batch, prec, dt):
    # 16 points up to 512 bytes are this kernel's, the others the compile-time
    # kernel's; a forced strategy keeps the latter at every length
    x = synth.uniform_complex(11 * n + batch, (batch, n), dt)
    short = 16 <= n <= (64 if prec == A.COMPLEX64 else 32)
    ref = O.fft_batch(x.astype(np.complex128))
    for strategy in (A.STRATEGY_AUTO, A.STRATEGY_STOCKHAM):
        with A.Plan.from_desc(ctx, (n,), precision=prec, batch=batch, strategy=strategy) as p:
            assert p.describe().startswith("hip_mixed") == (short and strategy == A.STRATEGY_AUTO)
            got = np.empty_like(x)
            p.forward(got, x)
            back = got.copy()
            p.inverse(back, back)   # in place
        assert rel_l2(got, ref) <= _tol(prec, n)
        assert rel_l2(back, O.fft_batch(got.astype(np.complex128), inverse=True)) <= _tol(prec, n)


# one-launch convolution forms of lengths with a prime factor above 7: Rader
# (n - 1 of one to four passes, the longest of either precision) and Bluestein
# with a padded length that is not a power of two; rows apart from each other,
# in place, partial groups, against a forced power-of-two-or-smooth Bluestein
@pytest.mark.parametrize("prec,dt", PRECS)
@pytest.mark.parametrize("n", [11, 13, 17, 19, 31, 71, 127, 257, 1009, 1459, 2017, 4051, 8101, 8641, 10369, 12289, 18433, 20161])
@pytest.mark.parametrize("gap", [0, 3])
def test_prime_rows(ctx, n, gap, prec, dt):
    if (n - 1) * (16 if prec else 8) > 163840:
        pytest.skip("longer rows take the three-pass chain")
    # enough rows for the one-launch form
    m = 1 << (2 * n - 2).bit_length()
    batch = (1 << 15) // m + 3 if m <= 128 else (1 << 22) // m + 3 if m <= 4096 else 67
    buf = synth.uniform_complex(n + gap, (batch, n + gap), dt)
    x = np.ascontiguousarray(buf[:, :n])
    ref = np.fft.fft(x.astype(np.complex128), axis=1)
    for strategy in (A.STRATEGY_AUTO, A.STRATEGY_BLUESTEIN):
        with A.Plan.from_desc(ctx, (n,), precision=prec, batch=batch, idist=n + gap, odist=n + gap,
                              strategy=strategy) as p:
            if strategy == A.STRATEGY_BLUESTEIN:
                assert p.describe().startswith(f"hip_bluestein{n}m")
            elif n - 1 <= (8192 if prec else 16384):
                assert p.describe() == f"hip_rader{n}"
            dx = torch.from_numpy(buf).cuda()
            dy = torch.full_like(dx, 7)
            s = torch.cuda.Stream()
            s.wait_stream(torch.cuda.current_stream())
            p.exec_device(A.FORWARD, dy.data_ptr(), dx.data_ptr(), s.cuda_stream)
            s.synchronize()
            got = dy.cpu().numpy()
            p.exec_device(A.INVERSE, dy.data_ptr(), dy.data_ptr(), s.cuda_stream)   # in place
            s.synchronize()
            back = dy.cpu().numpy()
        assert np.all(got[:, n:] == 7) and np.all(back[:, n:] == 7)
        assert rel_l2(got[:, :n], ref) <= _tol(prec, n)
        assert rel_l2(back[:, :n], np.fft.ifft(got[:, :n].astype(np.complex128), axis=1)) <= _tol(prec, n)


@pytest.mark.parametrize("prec,dt", PRECS)
@pytest.mark.parametrize("n", [22, 67, 69, 143, 341, 503, 703, 1111, 2053, 2587, 5117, 6002, 8209, 9797, 10201])
def test_bluestein_rows_padded_to_smooth_lengths(ctx, n, prec, dt):
    m = 1 << (2 * n - 2).bit_length()   # rows enough for the one-launch form
    batch = (1 << 24) // m + 3 if m <= 4096 else 515
    x = synth.uniform_complex(n, (batch, n), dt)
    with A.Plan.from_desc(ctx, (n,), precision=prec, batch=batch) as p:
        got = np.empty_like(x)
        p.forward(got, x)
        back = got.copy()
        p.inverse(back, back)
    assert rel_l2(got, np.fft.fft(x.astype(np.complex128), axis=1)) <= _tol(prec, n)
    assert rel_l2(back, np.fft.ifft(got.astype(np.complex128), axis=1)) <= _tol(prec, n)


# real rows of 32 and 64 points are this kernel's from 1024 rows on, their
# neighbours and fewer rows k_real's
@pytest.mark.parametrize("prec", [A.COMPLEX64, A.COMPLEX128])
@pytest.mark.parametrize("n", [16, 32, 64, 128])
@pytest.mark.parametrize("batch", [1, 67, 4099])
def test_short_power_of_two_real_rows(ctx, n, batch, prec):
    rdt, cdt = (np.float32, np.complex64) if prec == A.COMPLEX64 else (np.float64, np.complex128)
    x = synth.uniform_real(n + batch, (batch, n), rdt)
    with A.Plan.from_desc(ctx, (n,), precision=prec, kind=A.R2C, batch=batch) as p:
        X = np.empty((batch, n // 2 + 1), cdt)
        p.forward(X, x)
        y = np.empty_like(x)
        p.inverse(y, X)
    assert rel_l2(X, O.rfft(x.astype(np.float64))) <= _tol(prec, n)
    assert rel_l2(y, O.irfft(X.astype(np.complex128), n)) <= _tol(prec, n)


# long power-of-two columns: 128 side by side take one pass, fewer two
@pytest.mark.parametrize("prec,dt", PRECS)
@pytest.mark.parametrize("cols,pad", [(127, 0), (128, 0), (131, 0), (200, 5)])
@pytest.mark.parametrize("n", [2048, 4096])
def test_long_power_of_two_columns(ctx, n, cols, pad, prec, dt):
    w = cols + pad
    buf = synth.uniform_complex(n + cols, (n, w), dt)
    with A.Plan.from_desc(ctx, (n,), precision=prec, batch=cols, istride=w, idist=1, ostride=w, odist=1) as p:
        if n * buf.itemsize >= 32768:
            assert p.describe() == f"hip_mixed{n}c" if cols >= 128 else "colfourstep" in p.describe()
        out = np.zeros_like(buf)
        p.forward(out.ravel(), buf.ravel())
        back = out.copy()
        p.inverse(back.ravel(), back.ravel())   # in place
    ref = O.fft_batch(np.ascontiguousarray(buf[:, :cols].T).astype(np.complex128)).T
    assert rel_l2(out[:, :cols], ref) <= _tol(prec, n)
    assert rel_l2(back[:, :cols], buf[:, :cols]) <= 2 * _tol(prec, n)


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("direction", [A.FORWARD, A.INVERSE])
def test_spread_real_rows_over_the_next_row(ctx, direction, noalloc):
    """Rows far apart whose outputs lie over the next row's input: the copy
    holds the rows alone, so it fits the static scratch although the rows'
    extent (72 MB) does not."""
    import ctypes
    n, batch, pitch = 50, 300, 30000   # pitch in complex elements
    h = n // 2
    x = synth.uniform_real(n, (batch, n), np.float32)
    X = np.fft.rfft(x.astype(np.float64), axis=1)
    src = x.view(np.complex64) if direction == A.FORWARD else X.astype(np.complex64)
    buf = torch.zeros((batch + 1, pitch), dtype=torch.complex64, device="cuda")
    buf[:batch, :src.shape[1]] = torch.from_numpy(np.ascontiguousarray(src)).cuda()
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    fn = A.lib().afft_plan_exec_device_noalloc if noalloc else A.lib().afft_plan_exec_device
    with A.Plan.from_desc(ctx, (n,), kind=A.R2C, batch=batch, idist=2 * pitch, odist=pitch) as p:
        A.check(fn(p.h, direction, ctypes.c_void_p(buf[1:].data_ptr()), ctypes.c_void_p(buf.data_ptr()),
                   ctypes.c_void_p(s.cuda_stream)))
        s.synchronize()
    if direction == A.FORWARD:
        assert rel_l2(buf[1:, :h + 1].cpu().numpy(), X) <= c64_tol(n)
    else:
        assert rel_l2(np.ascontiguousarray(buf[1:, :h].cpu().numpy()).view(np.float32), x) <= 2 * c64_tol(n)


# single launches where other lengths go through scratch: dst over src with
# other distances between the rows or columns
@pytest.mark.parametrize("prec,dt", PRECS)
@pytest.mark.parametrize("kind", ["rows", "columns"])
@pytest.mark.parametrize("noalloc", [False, True])
def test_other_distances_over_the_input(ctx, kind, noalloc, prec, dt):
    import ctypes
    if kind == "rows":   # Rader's form, its power of two beyond LDS
        n, batch = (12289 if prec == A.COMPLEX64 else 4201), 70
        lay = dict(idist=n, odist=n + 5)
    else:
        n, batch = (4096 if prec == A.COMPLEX64 else 2048), 130
        lay = dict(istride=batch, idist=1, ostride=batch + 5, odist=1)
    x = synth.uniform_complex(n, (batch, n), dt)
    ref = np.fft.fft(x.astype(np.complex128), axis=1)
    buf = torch.zeros(batch * n + 5 * max(n, batch), dtype=torch.from_numpy(x[:1]).dtype, device="cuda")
    buf[:batch * n] = torch.from_numpy(np.ascontiguousarray(x if kind == "rows" else x.T).ravel()).cuda()
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    fn = A.lib().afft_plan_exec_device_noalloc if noalloc else A.lib().afft_plan_exec_device
    with A.Plan.from_desc(ctx, (n,), precision=prec, batch=batch, **lay) as p:
        assert p.describe() in (f"hip_rader{n}", f"hip_mixed{n}c")
        for i in range(2):
            A.check(fn(p.h, A.FORWARD if i == 0 else A.INVERSE, ctypes.c_void_p(buf.data_ptr()),
                       ctypes.c_void_p(buf.data_ptr()), ctypes.c_void_p(s.cuda_stream)))
            s.synchronize()
            if i == 0:
                y = buf.cpu().numpy()
                got = (y[:batch * (n + 5)].reshape(batch, n + 5)[:, :n] if kind == "rows"
                       else y[:n * (batch + 5)].reshape(n, batch + 5)[:, :batch].T)
                assert rel_l2(got, ref) <= _tol(prec, n)
                # the inverse reads the plan's input layout
                z = np.ascontiguousarray(got if kind == "rows" else got.T)
                buf[:batch * n] = torch.from_numpy(z.ravel()).cuda()
                torch.cuda.synchronize()
    y = buf.cpu().numpy()
    got = (y[:batch * (n + 5)].reshape(batch, n + 5)[:, :n] if kind == "rows"
           else y[:n * (batch + 5)].reshape(n, batch + 5)[:, :batch].T)
    assert rel_l2(got, x) <= 2 * _tol(prec, n)


# k_fft's planar exchanges (two blocks a CU and more) against numpy, the last
# block partial
@pytest.mark.parametrize("kind,n,prec", [("rows", 8192, A.COMPLEX128), ("columns", 1024, A.COMPLEX64),
                                         ("columns", 512, A.COMPLEX128)])
@pytest.mark.parametrize("direction", [A.FORWARD, A.INVERSE])
def test_planar_exchange(ctx, kind, n, prec, direction):
    dt = torch.complex64 if prec == A.COMPLEX64 else torch.complex128
    batch = 515 if kind == "rows" else 512 * 16 + 5   # 16 columns a block
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn((batch, n) if kind == "rows" else (n, batch), generator=g, device="cuda", dtype=dt)
    y = torch.empty_like(x)
    lay = {} if kind == "rows" else dict(istride=batch, idist=1, ostride=batch, odist=1)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with A.Plan.from_desc(ctx, (n,), precision=prec, batch=batch, **lay) as p:
        assert p.describe() == f"hip_lds{n}" + kind[0]
        p.exec_device(direction, y.data_ptr(), x.data_ptr(), s.cuda_stream)
        s.synchronize()
    fft = np.fft.fft if direction == A.FORWARD else np.fft.ifft
    ref = fft(x.cpu().numpy().astype(np.complex128), axis=1 if kind == "rows" else 0)
    got = y.cpu().numpy()
    assert rel_l2(got, ref) <= _tol(prec, n)
    if kind == "rows":
        assert rel_l2(got[-1], ref[-1]) <= _tol(prec, n)
    else:
        assert rel_l2(got[:, -5:], ref[:, -5:]) <= _tol(prec, n)
