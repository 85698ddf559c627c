"""Launch shapes that depend on how many transforms a plan has: rows of one
radix in two passes, columns and Rader rows a thread per butterfly where there
are few, and rough rows that stay on the compile-time kernel; against
numpy, within the library's budgets."""
import numpy as np
import pytest
import torch

import algofft_hip as A
from helpers import C128_TOL, c64_tol, rel_l2

pytestmark = pytest.mark.gpu

PRECS = [(A.COMPLEX64, torch.complex64), (A.COMPLEX128, torch.complex128)]


def _run(ctx, n, batch, prec, dt, columns=False):
    g = torch.Generator(device="cuda").manual_seed(n + batch)
    x = torch.randn((n, batch) if columns else (batch, n), generator=g, device="cuda", dtype=dt)
    y = torch.empty_like(x)
    lay = dict(istride=batch, idist=1, ostride=batch, odist=1) if columns else {}
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with A.Plan.from_desc(ctx, (n,), precision=prec, batch=batch, **lay) as p:
        algo = p.describe()
        p.exec_device(A.FORWARD, y.data_ptr(), x.data_ptr(), s.cuda_stream)
        s.synchronize()
    ref = np.fft.fft(x.cpu().numpy().astype(np.complex128), axis=0 if columns else 1)
    tol = c64_tol(n) if prec == A.COMPLEX64 else C128_TOL
    got = y.cpu().numpy()
    assert rel_l2(got, ref) <= tol
    edge = (slice(None), slice(-3, None)) if columns else slice(-3, None)
    assert rel_l2(got[edge], ref[edge]) <= 2 * tol
    return algo


@pytest.mark.parametrize("prec,dt", PRECS)
@pytest.mark.parametrize("n", [10, 14, 16, 18, 20])
@pytest.mark.parametrize("batch", [5, 4001, 120001])
def test_rows_of_one_radix(ctx, n, batch, prec, dt):
    _run(ctx, n, batch, prec, dt)


@pytest.mark.parametrize("prec,dt", PRECS)
@pytest.mark.parametrize("n", [11, 13, 17, 19])
@pytest.mark.parametrize("batch", [2001, 120001])
def test_rader_rows_of_one_radix(ctx, n, batch, prec, dt):
    _run(ctx, n, batch, prec, dt)


@pytest.mark.parametrize("prec,dt", PRECS)
@pytest.mark.parametrize("n,cols", [(49, 5), (625, 33), (625, 1500), (1225, 500), (2401, 33), (3125, 7), (4000, 130)])
def test_few_columns(ctx, n, cols, prec, dt):
    _run(ctx, n, cols, prec, dt, columns=True)


# many columns, blocks below half a CU's LDS
@pytest.mark.parametrize("n,cols", [(320, 4099), (640, 4099), (1280, 2051)])
def test_many_columns(ctx, n, cols):
    _run(ctx, n, cols, A.COMPLEX128, torch.complex128, columns=True)


# padded to 175 points in three passes these rows took 90 us where the two passes
# of 256 take 54
@pytest.mark.parametrize("n", [85, 86, 87, 88])
def test_rough_rows_on_two_passes_of_256(ctx, n):
    assert _run(ctx, n, 98689, A.COMPLEX64, torch.complex64) == f"hip_bluestein{n}m256"
