"""Rounding of the smooth four-step: its relative error is that of the two
passes' transforms, each measured as rows of its own, and of one product with a
factor that is rounded once, as independent contributions add."""
import numpy as np
import pytest

import algofft_hip as A
from algofft_hip import synth

pytestmark = pytest.mark.gpu


def _error(ctx, n, rows, **kw):
    x = synth.uniform_complex(n, (rows, n), np.complex64)
    with A.Plan.from_desc(ctx, (n,), batch=rows, **kw) as p:
        got = np.empty_like(x)
        p.forward(got, x)
    ref = np.fft.fft(x.astype(np.complex128), axis=1)
    return float(np.linalg.norm(got - ref) / np.linalg.norm(ref))


def _product_error():
    x = synth.uniform_complex(1, (100000,), np.complex64)
    w = np.exp(-2j * np.pi * np.arange(x.size) / x.size)
    w32 = w.astype(np.complex64)
    re = x.real * w32.real - x.imag * w32.imag
    im = x.real * w32.imag + x.imag * w32.real
    ref = x.astype(np.complex128) * w
    return float(np.linalg.norm((re + 1j * im) - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("n1,n2", [(125, 144), (120, 200), (150, 200), (200, 500)])
def test_error_of_the_passes_and_one_rounded_factor(ctx, n1, n2):
    whole = _error(ctx, n1 * n2, 8, strategy=A.STRATEGY_SIXSTEP, split=n1)
    parts = [_error(ctx, n, 160000 // n, strategy=A.STRATEGY_MIXED) for n in (n1, n2)] + [_product_error()]
    # a tenth for the passes' other radix orders in the two layouts
    assert whole <= 1.1 * float(np.linalg.norm(parts)), (whole, parts)
