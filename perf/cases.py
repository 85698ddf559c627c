"""Workloads whose time on the GPU is followed: what programs that use this
library ask of it, through its public Python entry points on device-resident
data.

Each kind of case stands for one use:

  c2c      batched, N-D or long complex transforms (Plan.exec_device)
  pair     a forward and an inverse transform of one small batch: the
           smallest calls, where launch latency counts
  r2c/c2r  real rows, images and volumes and their way back
  ragged   many transforms of mixed lengths as one graph (Ragged.exec_graph)
  conv     batched linear convolution (afft_conv_exec)
"""
import ctypes
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "algo-fft_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import algofft_hip as A  # noqa: E402
from algofft_hip import synth  # noqa: E402

_CONV_MODES = {"linear": A.CONV_LINEAR, "correlate": A.CONV_CORRELATE, "real": A.CONV_REAL}


def _c2c(name, dims, batch, direction="forward", precision=64):
    return {"name": name, "kind": "c2c", "dims": dims, "batch": batch, "direction": direction, "precision": precision}


def listed():
    return [
        # one short signal there and back (a filter step): two launches
        {"name": "pair_256", "kind": "pair", "dims": "256", "batch": 1, "precision": 64},
        # the benchmark's headline: a large batch of power-of-two rows
        _c2c("rows_pow2_4096", "4096", 16384),
        # the same amount of data at a length that is not a power of two
        # (7-smooth lengths are what callers pad or cut their signals to)
        _c2c("rows_smooth_3000", "3000", 22369),
        # long signals, beyond one block's local memory
        _c2c("long_pow2_1048576", "1048576", 64),
        _c2c("long_smooth_100000", "100000", 671, "inverse"),
        # lengths nobody chose: a prime, at an ordinary batch
        _c2c("rows_prime_1009", "1009", 8192),
        # a long prime in double precision
        _c2c("long_prime_1000003", "1000003", 8, precision=128),
        # double-precision grids: contiguous rows, then the strided axis
        _c2c("grid_1200x1500_c128", "1200x1500", 18, "inverse", precision=128),
        # a stack of real images (full-HD frames)
        {"name": "image_1080x1920", "kind": "r2c", "dims": "1080x1920", "batch": 16, "precision": 64},
        # a real volume brought back from its half spectrum
        {"name": "volume_512", "kind": "c2r", "dims": "512x512x512", "batch": 1, "precision": 64},
        # transforms of mixed lengths, as they arrive in a service's queue
        {"name": "ragged_4096", "kind": "ragged", "count": 4096, "lo": 16, "hi": 65536, "sizes_seed": 1234,
         "direction": "forward", "precision": 64},
        # real signals against a filter of a few taps
        {"name": "conv_real_1000x33", "kind": "conv", "na": 1000, "nb": 33, "batch": 16384, "mode": "real",
         "precision": 64},
    ]


# ---- drawn cases --------------------------------------------------------------

def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth(n):
    for q in (2, 3, 5, 7):
        while n % q == 0:
            n //= q
    return n == 1


def _near_smooth(v, step=1):
    v = max(step, v // step * step)
    while not _smooth(v):
        v += step
    return v


def _near_prime(v):
    v = max(11, v | 1)
    while any(v % q == 0 for q in range(3, int(v ** 0.5) + 1, 2)):
        v += 2
    return v


def _rough(rng, v):
    """A length with a prime factor above 7: a prime or a multiple of one."""
    if rng.random() < 0.5:
        return _near_prime(v)
    q = rng.choice([11, 13, 17, 19, 23, 31])
    return q * max(1, v // q)


def draw(rng):
    """One more case: any kind of the list, lengths and batches log-uniform
    over the ranges that the library covers, at most 2^26 complex64 (2^25
    complex128) points each way."""
    kind = rng.choice(["pair", "rows_pow2", "rows_smooth", "rows_smooth", "rows_rough", "long_pow2", "long_smooth",
                       "long_rough", "grid", "real", "real", "ragged", "conv", "conv"])
    precision = rng.choice([64, 64, 128])
    wide = 1 if precision == 64 else 2
    direction = rng.choice(["forward", "inverse"])
    cap = (16384 if precision == 64 else 8192)
    if kind == "pair":
        return {"kind": "pair", "dims": str(_near_smooth(_log_int(rng, 16, 4096))), "batch": _log_int(rng, 1, 64),
                "precision": precision}
    if kind.startswith("rows"):
        n = _log_int(rng, 16, cap)
        if kind == "rows_pow2":
            n = 1 << int(math.log2(n))
        elif kind == "rows_smooth":
            n = _near_smooth(n)
        else:
            n = _rough(rng, max(17, n // 2))
        total = _log_int(rng, 1 << 18, (1 << (24 if kind == "rows_rough" else 26)) // wide)
        return {"kind": "c2c", "dims": str(n), "batch": max(1, total // n), "direction": direction,
                "precision": precision}
    if kind.startswith("long"):
        n = _log_int(rng, cap + 1, 1 << (19 if kind == "long_rough" else 22))
        if kind == "long_pow2":
            n = 1 << int(math.ceil(math.log2(n)))
        elif kind == "long_smooth":
            n = _near_smooth(n)
        else:
            n = _rough(rng, n)
        total = _log_int(rng, n, (1 << (23 if kind == "long_rough" else 26)) // wide)
        return {"kind": "c2c", "dims": str(n), "batch": max(1, total // n), "direction": direction,
                "precision": precision}
    if kind == "grid":
        rank = rng.choice([2, 2, 3])
        top = 4096 if rank == 2 else 256
        side = [_log_int(rng, 24, top) for _ in range(rank)]
        side = [(1 << int(math.log2(v))) if rng.random() < 0.4 else _near_smooth(v) for v in side]
        total = _log_int(rng, 1 << 20, (1 << 26) // wide)
        return {"kind": "c2c", "dims": "x".join(map(str, side)), "batch": max(1, total // math.prod(side)),
                "direction": direction, "precision": precision}
    if kind == "real":
        rank = rng.choice([1, 2, 2, 3])
        top = {1: 16384, 2: 4096, 3: 256}[rank]
        side = [_log_int(rng, 24, top) for _ in range(rank)]
        side = [(1 << int(math.log2(v))) if rng.random() < 0.4 else _near_smooth(v, 2) for v in side]
        total = _log_int(rng, 1 << 20, (1 << 26) // wide)
        return {"kind": rng.choice(["r2c", "c2r"]), "dims": "x".join(map(str, side)),
                "batch": max(1, total // math.prod(side)), "precision": precision}
    if kind == "ragged":
        return {"kind": "ragged", "count": _log_int(rng, 64, 4096), "lo": 16, "hi": _log_int(rng, 2048, 65536),
                "sizes_seed": rng.randrange(1 << 30), "direction": direction, "precision": precision}
    na = _log_int(rng, 64, 16384)
    nb = _log_int(rng, 9, na)
    total = _log_int(rng, 1 << 18, (1 << 24) // wide)
    return {"kind": "conv", "na": na, "nb": nb, "batch": max(1, total // (na + nb)),
            "mode": rng.choice(["linear", "correlate", "real"]), "precision": precision}


# ---- a program's state ----------------------------------------------------------

_program = {}


def _ctx():
    """A program opens the device once and enqueues on a stream of its own."""
    if not _program:
        _program["ctx"] = A.Context(0)
        _program["stream"] = torch.cuda.Stream()
    return _program["ctx"], _program["stream"]


class _State(dict):
    """Buffers and the plan of one case; the plan is closed with it."""

    def __del__(self):
        close = self.pop("close", None)
        if close:
            try:
                close()
            except Exception:   # interpreter shutdown
                pass


def _dims(case):
    return tuple(int(v) for v in case["dims"].split("x"))


def _types(case):
    wide = case["precision"] == 128
    return ((A.COMPLEX128, torch.complex128, torch.float64) if wide else (A.COMPLEX64, torch.complex64, torch.float32))


def _signal(seed, shape, dtype):
    """Noise with a few strong tones along the last axis, as measured signals
    and spectra have (dynamic range about 1e3)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    real = torch.float64 if dtype in (torch.complex128, torch.float64) else torch.float32
    x = torch.randn(tuple(shape), generator=g, device="cuda", dtype=dtype)
    n = shape[-1]
    t = torch.arange(n, device="cuda", dtype=torch.int64)
    for k in range(3):
        f = int(torch.randint(n, (1,), generator=g, device="cuda"))
        ph = (f * t % n).to(torch.float64) * (2 * math.pi / n)
        tone = torch.polar(torch.full_like(ph, 3.0 / (k + 1)), ph)
        x += tone.to(dtype) if dtype.is_complex else tone.real.to(real)
    return x


def _ragged_sizes(case):
    return synth.ragged_sizes(case["sizes_seed"], case["count"], case["lo"], case["hi"])


def _inputs(case, seed):
    prec, ctype, rtype = _types(case)
    kind = case["kind"]
    if kind == "ragged":
        return _signal(seed, (sum(_ragged_sizes(case)),), ctype)
    if kind == "conv":
        dtype = rtype if case["mode"] == "real" else ctype
        return (_signal(seed, (case["batch"], case["na"]), dtype),
                _signal(seed + 1000003, (case["batch"], case["nb"]), dtype))
    shape = (case["batch"],) + _dims(case)
    if kind == "c2r":
        return _half_spectrum(_signal(seed, shape, rtype))
    return _signal(seed, shape, rtype if kind == "r2c" else ctype)


def _half_spectrum(x):
    """A valid half spectrum (Hermitian where it has to be) made of the even
    and odd parts of x under k -> -k along every axis."""
    flip = x
    for ax in range(1, x.dim()):
        flip = torch.roll(torch.flip(flip, (ax,)), 1, ax)
    h = x.shape[-1] // 2 + 1
    return torch.complex((x + flip)[..., :h].contiguous(), (x - flip)[..., :h].contiguous())


def prepare(case, seed):
    ctx, stream = _ctx()
    prec, ctype, rtype = _types(case)
    kind = case["kind"]
    x = _inputs(case, seed)
    st = _State(kind=kind, stream=stream.cuda_stream, x=x)
    if kind == "ragged":
        rg = A.Ragged(ctx, _ragged_sizes(case), prec)
        st.update(ragged=rg, close=rg.close, y=torch.empty_like(x))
    elif kind == "conv":
        h = ctypes.c_void_p()
        A.check(A.lib().afft_conv_create(ctx.h, prec, case["na"], case["nb"], case["batch"],
                                         _CONV_MODES[case["mode"]], ctypes.byref(h)))
        st.update(conv=h, close=lambda: A.lib().afft_conv_destroy(h),
                  y=torch.empty((case["batch"], case["na"] + case["nb"] - 1), dtype=x[0].dtype, device="cuda"))
    else:
        dims = _dims(case)
        plan = A.Plan.from_desc(ctx, dims, precision=prec, batch=case["batch"],
                                kind={"c2c": A.C2C, "pair": A.C2C, "r2c": A.R2C, "c2r": A.C2R}[kind])
        st.update(plan=plan, close=plan.close)
        if kind == "r2c":
            st["y"] = torch.empty((case["batch"],) + dims[:-1] + (dims[-1] // 2 + 1,), dtype=ctype, device="cuda")
        elif kind == "c2r":
            st["y"] = torch.empty((case["batch"],) + dims, dtype=rtype, device="cuda")
        else:
            st["y"] = torch.empty_like(x)
        if kind == "pair":
            st["z"] = torch.empty_like(x)
    inverse = kind == "c2r" or case.get("direction") == "inverse"
    st["direction"] = A.INVERSE if inverse else A.FORWARD
    torch.cuda.synchronize()
    return st


def run(state):
    kind, s, x, y = state["kind"], state["stream"], state["x"], state["y"]
    if kind == "ragged":
        state["ragged"].exec_graph(state["direction"], y.data_ptr(), x.data_ptr(), s)
    elif kind == "conv":
        A.check(A.lib().afft_conv_exec(state["conv"], ctypes.c_void_p(y.data_ptr()), ctypes.c_void_p(x[0].data_ptr()),
                                       ctypes.c_void_p(x[1].data_ptr()), ctypes.c_void_p(s)))
    elif kind == "pair":
        z = state["z"]
        state["plan"].exec_device(A.FORWARD, y.data_ptr(), x.data_ptr(), s)
        state["plan"].exec_device(A.INVERSE, z.data_ptr(), y.data_ptr(), s)
        return {"spectrum": y, "signal": z}
    else:
        state["plan"].exec_device(state["direction"], y.data_ptr(), x.data_ptr(), s)
    return y


# ---- what a pass cannot do without ------------------------------------------------

def _fft_flops(n):
    return 5.0 * n * math.log2(max(2, n))


def work(case):
    es = 16 if case["precision"] == 128 else 8
    kind = case["kind"]
    if kind == "ragged":
        sizes = _ragged_sizes(case)
        return {"bytes": 2 * es * sum(sizes), "flops": sum(_fft_flops(n) for n in sizes)}
    if kind == "conv":
        na, nb, b = case["na"], case["nb"], case["batch"]
        length = na + nb - 1
        half = 2 if case["mode"] == "real" else 1
        return {"bytes": es // half * b * (na + nb + length),
                "flops": b * (3 * _fft_flops(length) + 6 * length) / half}
    dims = _dims(case)
    n = math.prod(dims)
    b = case["batch"]
    if kind in ("r2c", "c2r"):
        hn = n // dims[-1] * (dims[-1] // 2 + 1)
        return {"bytes": b * (es // 2 * n + es * hn), "flops": b * _fft_flops(n) / 2}
    passes = 2 if kind == "pair" else 1
    return {"bytes": passes * 2 * es * n * b, "flops": passes * b * _fft_flops(n)}


# ---- the same in 64 bits -----------------------------------------------------------

def exact(case, seed):
    kind = case["kind"]
    x = _inputs(case, seed)
    if kind == "conv":
        a, b = (v.cpu().to(torch.complex128) for v in x)
        if case["mode"] == "correlate":
            b = torch.conj(torch.flip(b, (1,))).resolve_conj()
        length = case["na"] + case["nb"] - 1
        f = 1 << (length - 1).bit_length() if length > 1 else 1
        y = torch.fft.ifft(torch.fft.fft(a, n=f) * torch.fft.fft(b, n=f))[:, :length]
        return (y.real if case["mode"] == "real" else y).contiguous()
    inverse = case.get("direction") == "inverse"
    if kind == "ragged":
        v = x.cpu().to(torch.complex128)
        y = torch.empty_like(v)
        at = 0
        for n in _ragged_sizes(case):
            y[at:at + n] = (torch.fft.ifft if inverse else torch.fft.fft)(v[at:at + n])
            at += n
        return y
    dims = _dims(case)
    axes = tuple(range(1, len(dims) + 1))
    if kind == "r2c":
        return torch.fft.rfftn(x.cpu().to(torch.float64), dim=axes)
    if kind == "c2r":
        return torch.fft.irfftn(x.cpu().to(torch.complex128), s=dims, dim=axes)
    v = x.cpu().to(torch.complex128)
    if kind == "pair":
        return {"spectrum": torch.fft.fft(v), "signal": v}
    return (torch.fft.ifftn if inverse else torch.fft.fftn)(v, dim=axes)
