"""Normalised (1/N) and unitary (1/sqrt(N)) forward transforms on every
route of a complex plan: powers of two in one pass and in two, smooth lengths
in one pass and in two, the one-launch forms of rough lengths, the
three-pass Bluestein chain, rows and strided columns; against numpy, within the
library's budgets."""
import numpy as np
import pytest

import algofft_hip as A
from algofft_hip import synth
from helpers import C128_TOL, c64_tol, rel_l2

pytestmark = pytest.mark.gpu

# (n, rows): the last four are chains (few rows beyond LDS, a length beyond it)
ROUTES = [(16, 3), (256, 3), (4096, 130), (65536, 2), (3000, 3), (100000, 2), (17, 5), (341, 3), (1009, 70), (4099, 64),
          (4099, 1), (8209, 2), (12289, 3), (100003, 2)]


@pytest.mark.parametrize("prec,dt", [(A.COMPLEX64, np.complex64), (A.COMPLEX128, np.complex128)])
@pytest.mark.parametrize("flag", [A.FLAG_NORMALIZE, A.FLAG_UNITARY])
@pytest.mark.parametrize("columns", [False, True])
@pytest.mark.parametrize("n,rows", ROUTES)
def test_scaled_forward(ctx, n, rows, columns, flag, prec, dt):
    x = synth.uniform_complex(n + rows, (rows, n), dt)
    src = np.ascontiguousarray(x.T if columns else x)
    lay = dict(istride=rows, idist=1, ostride=rows, odist=1) if columns else {}
    got = np.empty_like(src)
    with A.Plan.from_desc(ctx, (n,), precision=prec, batch=rows, flags=flag, **lay) as p:
        p.forward(got.ravel(), src.ravel())
        back = np.empty_like(src)
        p.inverse(back.ravel(), got.ravel())   # the inverse carries 1/N whatever the forward does
    scale = 1.0 / n if flag == A.FLAG_NORMALIZE else 1.0 / np.sqrt(n)
    tol = c64_tol(n) if prec == A.COMPLEX64 else C128_TOL
    ref = np.fft.fft(x.astype(np.complex128), axis=1) * scale
    assert rel_l2(got.T if columns else got, ref) <= tol
    assert rel_l2(back.T if columns else back, x * scale) <= 2 * tol
