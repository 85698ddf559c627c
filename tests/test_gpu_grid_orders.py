"""Grids on both sides of the rules for their columns' block order and for rows of
64 points: sizes that the caches hold and larger ones, columns on line
boundaries and off them, one group of columns and several; against
numpy, within the library's budgets."""
import numpy as np
import pytest
import torch

import algofft_hip as A
from helpers import C128_TOL, c64_tol, rel_l2

pytestmark = pytest.mark.gpu

GRIDS = [((16, 8), 67), ((8, 32), 4096), ((8, 8, 128), 128), ((64, 64), 1024), ((64, 64), 2100), ((16, 64), 40), ((64, 100), 33),
         ((16, 64), 4100), ((64, 64, 64), 3)]


@pytest.mark.parametrize("prec,dt", [(A.COMPLEX64, torch.complex64), (A.COMPLEX128, torch.complex128)])
@pytest.mark.parametrize("dims,batch", GRIDS)
@pytest.mark.parametrize("direction", [A.FORWARD, A.INVERSE])
def test_grids(ctx, dims, batch, direction, prec, dt):
    g = torch.Generator(device="cuda").manual_seed(batch)
    x = torch.randn((batch,) + dims, generator=g, device="cuda", dtype=dt)
    y = torch.empty_like(x)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with A.Plan.from_desc(ctx, dims, precision=prec, batch=batch) as p:
        p.exec_device(direction, y.data_ptr(), x.data_ptr(), s.cuda_stream)
        s.synchronize()
    fft = np.fft.fftn if direction == A.FORWARD else np.fft.ifftn
    pick = [0, batch // 2, batch - 1]
    ref = fft(x[pick].cpu().numpy().astype(np.complex128), axes=tuple(range(1, len(dims) + 1)))
    tol = c64_tol(int(np.prod(dims))) if prec == A.COMPLEX64 else C128_TOL
    assert rel_l2(y[pick].cpu().numpy(), ref) <= tol
