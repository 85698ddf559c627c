"""The one-launch convolutions (kconv.hpp, kshort.hpp) over batches: shortest and
longest padded lengths, the first beyond them (the launches of their own),
partial groups, odd and one-element rows, and an output over an input;
against FP64 FFT convolution, within the library's budgets."""
import ctypes

import numpy as np
import pytest
import torch

import algofft_hip as A
from algofft_hip import synth
from helpers import C128_TOL, c64_tol, rel_l2

pytestmark = pytest.mark.gpu

# (na, nb, batch): complex cap 16384 (complex64) / 8192 padded points, real
# rows twice that
SHAPES = [(1, 1, 5), (2, 1, 3), (3, 4, 67), (7, 5, 33), (100, 29, 41), (777, 65, 32), (1009, 1009, 5), (4000, 93, 3),
          (5000, 3193, 2), (8000, 400, 2), (9000, 7300, 2), (16000, 16001, 1), (20000, 13000, 1)]


def _ref(a, b, mode):
    if mode == A.CONV_CORRELATE:
        b = np.conj(b[:, ::-1])
    n = a.shape[1] + b.shape[1] - 1
    f = 1 << int(np.ceil(np.log2(max(n, 2))))
    y = np.fft.ifft(np.fft.fft(a, f, axis=1) * np.fft.fft(b, f, axis=1), axis=1)[:, :n]
    return y.real if mode == A.CONV_REAL else y


def _run(ctx, prec, mode, na, nb, batch, dst, a, b):
    h = ctypes.c_void_p()
    A.check(A.lib().afft_conv_create(ctx.h, prec, na, nb, batch, mode, ctypes.byref(h)))
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    try:
        A.check(A.lib().afft_conv_exec(h, ctypes.c_void_p(dst.data_ptr()), ctypes.c_void_p(a.data_ptr()),
                                       ctypes.c_void_p(b.data_ptr()), ctypes.c_void_p(s.cuda_stream)))
        s.synchronize()
    finally:
        A.check(A.lib().afft_conv_destroy(h))


def _data(prec, mode, na, nb, batch):
    wide = prec == A.COMPLEX128
    if mode == A.CONV_REAL:
        dt = np.float64 if wide else np.float32
        return synth.uniform_real(na, (batch, na), dt), synth.uniform_real(nb + 7, (batch, nb), dt)
    dt = np.complex128 if wide else np.complex64
    return synth.uniform_complex(na, (batch, na), dt), synth.uniform_complex(nb + 7, (batch, nb), dt)


@pytest.mark.parametrize("na,nb,batch", SHAPES)
@pytest.mark.parametrize("mode", [A.CONV_LINEAR, A.CONV_CORRELATE, A.CONV_REAL])
@pytest.mark.parametrize("prec", [A.COMPLEX64, A.COMPLEX128])
def test_batched_convolution(ctx, na, nb, batch, mode, prec):
    a, b = _data(prec, mode, na, nb, batch)
    ta, tb = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    out = torch.empty((batch, na + nb - 1), dtype=ta.dtype, device="cuda")
    _run(ctx, prec, mode, na, nb, batch, out, ta, tb)
    tol = c64_tol(na + nb) if prec == A.COMPLEX64 else C128_TOL
    wide = np.float64 if mode == A.CONV_REAL else np.complex128
    assert rel_l2(out.cpu().numpy(), _ref(a.astype(wide), b.astype(wide), mode)) <= tol


@pytest.mark.parametrize("mode", [A.CONV_LINEAR, A.CONV_REAL])
@pytest.mark.parametrize("over", ["a", "b"])
def test_output_over_an_input(ctx, mode, over):
    na, nb, batch = 300, 45, 37
    a, b = _data(A.COMPLEX64, mode, na, nb, batch)
    big, small = (a, b) if over == "a" else (b, a)
    buf = torch.zeros(batch * (na + nb - 1), dtype=torch.from_numpy(a).dtype, device="cuda")
    buf[:big.size] = torch.from_numpy(big.ravel()).cuda()
    t = torch.from_numpy(small).cuda()
    ta, tb = (buf, t) if over == "a" else (t, buf)
    _run(ctx, A.COMPLEX64, mode, na, nb, batch, buf, ta, tb)
    wide = np.float64 if mode == A.CONV_REAL else np.complex128
    got = buf.cpu().numpy().reshape(batch, na + nb - 1)
    assert rel_l2(got, _ref(a.astype(wide), b.astype(wide), mode)) <= c64_tol(na + nb)


# the direct form (kshort.hpp): its longest taps and one more, on either side,
# tiles of 2304 (real) and 1792 (complex) outputs filled exactly, one over and
# one under, rows of every remainder of a thread's outputs, one tap
DIRECT = [(1, 1, 7), (5, 1, 300), (1, 5, 3), (13, 3, 100), (20, 7, 61), (40, 40, 9), (48, 48, 5), (49, 49, 5),
          (2209, 96, 3), (2210, 96, 3), (2208, 97, 2), (1745, 48, 3), (1746, 48, 2), (48, 1744, 2), (96, 5000, 2),
          (30000, 128, 1), (128, 40001, 1), (30000, 129, 1)]


@pytest.mark.parametrize("na,nb,batch", DIRECT)
@pytest.mark.parametrize("mode", [A.CONV_LINEAR, A.CONV_CORRELATE, A.CONV_REAL])
@pytest.mark.parametrize("prec", [A.COMPLEX64, A.COMPLEX128])
def test_short_sides(ctx, na, nb, batch, mode, prec):
    a, b = _data(prec, mode, na, nb, batch)
    ta, tb = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    out = torch.full((batch * (na + nb - 1) + 5,), 7, dtype=ta.dtype, device="cuda")
    _run(ctx, prec, mode, na, nb, batch, out, ta, tb)
    got = out.cpu().numpy()
    tol = c64_tol(na + nb) if prec == A.COMPLEX64 else C128_TOL
    assert np.all(got[-5:] == 7)
    assert rel_l2(got[:-5].reshape(batch, -1), _ref(a, b, mode)) <= tol


# the direct form's rounding: a box filter over constant rows, where every
# partial sum rounds alike.  With nonnegative terms each output is off by at most
# one unit roundoff per addition on the way to it: 4 products of a side in
# turn (2 taps' worth of either part for complex rows), the pair of them, 4 such
# blocks, the groups of these.
@pytest.mark.parametrize("taps,na", [(4, 100), (8, 200), (33, 1000), (48, 1000), (96, 1000), (128, 40000)])
@pytest.mark.parametrize("mode", [A.CONV_LINEAR, A.CONV_REAL])
@pytest.mark.parametrize("prec", [A.COMPLEX64, A.COMPLEX128])
def test_box_filter_over_constant_rows(ctx, taps, na, mode, prec):
    real = mode == A.CONV_REAL
    if taps > 48 and not real and na < 16384:
        pytest.skip("taken by the transforms")
    half = 4 if real else 2   # taps summed in turn
    depth = (min(taps, half) + (taps > half) + min(-(-taps // (2 * half)), 4) - 1 + -(-taps // (8 * half)) - 1) * (1 if real else 2)
    u = 2.0 ** -24 if prec == A.COMPLEX64 else 2.0 ** -53
    rdt = np.float32 if prec == A.COMPLEX64 else np.float64
    dt = rdt if real else (np.complex64 if prec == A.COMPLEX64 else np.complex128)
    c = np.concatenate([np.linspace(1, 2, 60), [1.9296482, 1.8442211, 1.0653267]]).astype(rdt)
    h = rdt(1.0 / taps)
    a = np.repeat(c[:, None], na, axis=1).astype(dt)
    b = np.full((len(c), taps), h, dt)
    ta, tb = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    out = torch.empty((len(c), na + taps - 1), dtype=ta.dtype, device="cuda")
    _run(ctx, prec, mode, na, taps, len(c), out, ta, tb)
    got = out.cpu().numpy()[:, taps - 1:na].real
    ref = (c.astype(np.longdouble) * np.longdouble(h) * taps)[:, None]
    assert float(np.max(np.abs(got - ref) / ref)) <= depth * u
