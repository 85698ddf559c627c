"""Creating a plan of a rough length looks at many padded lengths: those that no
launch shape holds are turned down without listing their radix orders.  Bound:
twenty times the 3 ms that such a plan takes; a full listing takes 90 ms and more
at some lengths."""
import time

import pytest

import algofft_hip as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,prec", [(9001, A.COMPLEX64), (10007, A.COMPLEX64), (9174, A.COMPLEX64),
                                    (4574, A.COMPLEX128), (4449, A.COMPLEX128)])
def test_rough_lengths_are_planned_quickly(ctx, n, prec):
    best = 1e9
    for _ in range(4):
        t = time.perf_counter()
        with A.Plan.from_desc(ctx, (n,), precision=prec, batch=300):
            best = min(best, time.perf_counter() - t)
    assert best < 0.06
