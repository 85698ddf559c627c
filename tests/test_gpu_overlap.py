"""Plans that read a copy of their input where dst overlaps it: a call over the
input leaves what later calls need as it was, and one may be captured after an
execution on separate buffers."""
import ctypes

import numpy as np
import pytest
import torch

import algofft_hip as A
from algofft_hip import synth
from helpers import c64_tol, rel_l2

pytestmark = pytest.mark.gpu


def _exec(p, direction, dst, src, stream, noalloc=False):
    fn = A.lib().afft_plan_exec_device_noalloc if noalloc else A.lib().afft_plan_exec_device
    return fn(p.h, direction, ctypes.c_void_p(dst.data_ptr()), ctypes.c_void_p(src.data_ptr()),
              ctypes.c_void_p(stream.cuda_stream))


@pytest.mark.parametrize("first", ["noalloc", "device"])
def test_a_call_over_its_input_leaves_separate_buffers_scratch_free(ctx, first):
    # packed real rows: the copy (65 MiB) does not fit the static scratch, and
    # separate buffers need none
    n, batch = 1920, 8800
    x = torch.from_numpy(synth.uniform_real(3, (batch, n), np.float32)).cuda()
    y = torch.empty((batch, n // 2 + 1), dtype=torch.complex64, device="cuda")
    over = torch.zeros(batch * (n + 2), dtype=torch.float32, device="cuda")
    over[:x.numel()] = x.ravel()
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with A.Plan.from_desc(ctx, (n,), kind=A.R2C, batch=batch) as p:
        held = p.workspace_bytes()
        assert held >= batch * n * 4 > A.lib().afft_noalloc_scratch_bytes()
        if first == "noalloc":
            assert _exec(p, A.FORWARD, over, over, s, noalloc=True) != A.OK
        else:
            A.check(_exec(p, A.FORWARD, over, over, s))
        A.check(_exec(p, A.FORWARD, y, x, s, noalloc=True))
        s.synchronize()
        assert p.workspace_bytes() == held
    ref = np.fft.rfft(x[-3:].cpu().numpy().astype(np.float64), axis=1)
    assert rel_l2(y[-3:].cpu().numpy(), ref) <= c64_tol(n)
    if first == "device":
        got = torch.view_as_complex(over.view(-1, 2)).view(batch, -1)[-3:].cpu().numpy()
        assert rel_l2(got, ref) <= c64_tol(n)


@pytest.mark.parametrize("kind", ["real rows", "rows", "columns"])
def test_capture_over_the_input_after_separate_buffers(ctx, kind):
    if kind == "real rows":
        n, batch, desc = 50, 37, dict(kind=A.R2C)
    elif kind == "rows":     # Rader's form, its power of two beyond LDS
        n, batch = 12289, 70
        desc = dict(idist=n, odist=n + 5)
    else:
        n, batch = 4096, 130
        desc = dict(istride=batch, idist=1, ostride=batch + 5, odist=1)
    with A.Plan.from_desc(ctx, (n,), batch=batch, **desc) as p:
        ni, no = p.io_len(A.FORWARD)
        if kind == "real rows":
            x = torch.from_numpy(synth.uniform_real(5, ni, np.float32)).cuda()
            no *= 2   # in reals
        else:
            x = torch.from_numpy(synth.uniform_complex(5, ni, np.complex64)).cuda()
        apart, over = (torch.zeros(max(ni, no), dtype=x.dtype, device="cuda") for _ in range(2))
        s = torch.cuda.Stream()
        torch.cuda.synchronize()
        A.check(_exec(p, A.FORWARD, apart, x, s))
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            rc = _exec(p, A.FORWARD, over, over, s)
        A.check(rc)
        for _ in range(3):   # eager work and a wait between the replays
            over.zero_()
            over[:ni] = x
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            at = torch.arange(no, device="cuda")
            if kind == "rows":
                at = at[at % (n + 5) < n]
            elif kind == "columns":
                at = at[at % (batch + 5) < batch]
            assert torch.equal(over[at], apart[at])
