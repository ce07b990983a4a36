"""The workloads on which the speed of this library is followed.

A case is a dict of plain values: the entry point ("kind"), its sizes and its
options.  `prepare` makes what a program has in hand before the call (inputs
on the GPU, plans, layers, output buffers), `run` is one pass through the
public entry points, `exact` the same outputs in 64 bits from torch.fft, and
`work` the bytes and operations that no implementation avoids.

Kinds:
  fft      torch_fft.fft / fft_adjoint of [batch, n, 2] fp16, optionally with its backward pass
  dropin   Plan1D / Plan2D.exec, the reference's call: in place on a buffer in
           digit-reversed order.  The caller keeps its input and transforms a
           copy of it, so that a pass can be repeated on finite values.
  natural  Plan1D / Plan2D.exec_natural, out of place
  fft32    torch_fft.fft32 / fft32_adjoint of [batch, n] complex64
  split    Plan2D.exec_split of FP32 images
  rfft     torch_fft.rfft of [batch, n] fp16 reals, optionally with its backward pass
  c2r      torch_fft.c2r of [batch, n/2 + 1, 2]
  uneven   MultiPlan.exec_natural over signals of mixed sizes
  conv     FFTConv1d on [batch, channels, n, 2]: forward, or a training step's
           forward and both gradients
"""
from __future__ import annotations

import math
import random

import torch

from tcfft_amd import FORWARD, INVERSE, MultiPlan, Plan1D, Plan2D, gen_rev, torch_fft

DEV = "cuda"


def listed():
    return [
        # One short call of an interactive program: launch and host latency.
        dict(name="fft_small", kind="fft", n=1024, batch=8, inverse=False, grad=False),
        # The benchmark's 4096 x 1024 batch through the reference's in-place call.
        dict(name="dropin_4096_b1024", kind="dropin", nx=0, n=4096, batch=1024, inverse=False),
        # The benchmark's headline batch through the same call.
        dict(name="dropin_65536_b256", kind="dropin", nx=0, n=65536, batch=256, inverse=False),
        # A spectral loss on long signals: forward and backward, a ragged batch.
        dict(name="fft_65536_grad", kind="fft", n=65536, batch=201, inverse=False, grad=True),
        # Long records of 2^20 samples back to the time domain (two passes).
        dict(name="natural_1m_b16", kind="natural", nx=0, n=1 << 20, batch=16, inverse=True),
        # Image filtering on the benchmark's 1024 x 1024 images.
        dict(name="natural_2d_1024", kind="natural", nx=1024, n=1024, batch=8, inverse=False),
        # complex64 spectra of ordinary frames, where fp16 is too coarse.
        dict(name="fft32_4096", kind="fft32", n=4096, batch=3000, inverse=False, grad=False),
        # The benchmark's split-precision batch, with the adjoint as its backward.
        dict(name="fft32_65536_grad", kind="fft32", n=65536, batch=128, inverse=False, grad=True),
        # FP32 images at near-FP32 accuracy.
        dict(name="split_2d_1024", kind="split", nx=1024, n=1024, batch=8, inverse=True),
        # Real audio-like frames through a spectral layer and back.
        dict(name="rfft_8192_grad", kind="rfft", n=8192, batch=4099, grad=True),
        # Signals of many lengths in one launch (the benchmark's size mix).
        dict(name="uneven_2048", kind="uneven", signals=2048, mix=1, inverse=False),
        # A training step of the benchmark's long-convolution layer.
        dict(name="conv_train_8192", kind="conv", n=8192, channels=256, batch=32, grad=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """Sizes spread over the logarithm of the ranges, batches of any number."""
    kind = rng.choice(["fft", "fft", "dropin", "natural", "natural2d", "dropin2d", "fft32", "fft32", "split",
                       "rfft", "c2r", "uneven", "conv"])
    most = 1 << 24  # complex points of the largest drawn pass
    inverse = rng.random() < 0.4
    grad = rng.random() < 0.4
    if kind in ("fft", "dropin", "natural"):
        n = 1 << rng.randint(8, 22)
        c = dict(kind=kind, n=n, batch=_log_int(rng, 1, most // n), inverse=inverse)
        return dict(c, grad=grad) if kind == "fft" else dict(c, nx=0)
    if kind in ("natural2d", "dropin2d", "split"):
        n, nx = 1 << rng.randint(8, 12), 1 << rng.randint(5, 11)
        top = most // (1 if kind != "split" else 2)
        return dict(kind=kind.replace("2d", ""), nx=nx, n=n, batch=_log_int(rng, 1, max(1, top // (n * nx))),
                    inverse=inverse)
    if kind == "fft32":
        n = 1 << rng.randint(8, 20)
        return dict(kind=kind, n=n, batch=_log_int(rng, 1, most // 2 // n), inverse=inverse, grad=grad)
    if kind == "rfft":
        n = 1 << rng.randint(9, 20)
        return dict(kind=kind, n=n, batch=_log_int(rng, 1, 2 * most // n), grad=grad)
    if kind == "c2r":
        n = 1 << rng.randint(9, 20)
        return dict(kind=kind, n=n, batch=_log_int(rng, 1, 2 * most // n))
    if kind == "uneven":
        return dict(kind=kind, signals=_log_int(rng, 16, 1100), mix=rng.randint(2, 1 << 20), inverse=inverse)
    n, channels = 1 << rng.randint(11, 15), _log_int(rng, 3, 96)
    return dict(kind=kind, n=n, channels=channels, batch=_log_int(rng, 1, max(1, most // (n * channels))), grad=grad)


def _sizes(case):
    """Signal lengths 2^8 .. 2^16, evenly by exponent (a property of the case)."""
    r = random.Random(case["mix"])
    return [1 << r.randint(8, 16) for _ in range(case["signals"])]


def _rand(gen, *shape, dtype=torch.float16):
    """Uniform [-1, 1), the range of the reference's generator."""
    return (torch.rand(*shape, generator=gen, device=DEV) * 2 - 1).to(dtype)


def _inputs(case, seed):
    """The tensors made from the seed, in natural order."""
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    kind = case["kind"]
    if kind == "uneven":
        return {"x": _rand(gen, sum(_sizes(case)), 2)}
    n, batch = case["n"], case["batch"]
    if kind in ("fft", "dropin", "natural"):
        shape = (batch, n, 2) if not case.get("nx") else (batch, case["nx"], n, 2)
        t = {"x": _rand(gen, *shape)}
        if case.get("grad"):
            t["gy"] = _rand(gen, *shape)
        return t
    if kind == "fft32":
        t = {"x": torch.view_as_complex(_rand(gen, batch, n, 2, dtype=torch.float32))}
        if case["grad"]:
            t["gy"] = torch.view_as_complex(_rand(gen, batch, n, 2, dtype=torch.float32))
        return t
    if kind == "split":
        return {"x": _rand(gen, batch, case["nx"], n, 2, dtype=torch.float32)}
    if kind == "rfft":
        t = {"x": _rand(gen, batch, n)}
        if case["grad"]:
            t["gy"] = _rand(gen, batch, n // 2 + 1, 2)
        return t
    if kind == "c2r":
        return {"x": _rand(gen, batch, n // 2 + 1, 2)}
    if kind == "conv":
        t = {"x": _rand(gen, batch, case["channels"], n, 2),
             "h": torch.randn(case["channels"], n, 2, generator=gen, device=DEV) * 0.02}
        if case["grad"]:
            t["gy"] = _rand(gen, batch, case["channels"], n, 2)
        return t
    raise ValueError(kind)


def _reversal(radices, n):
    return torch.as_tensor(gen_rev(n, radices).astype("int64"), device=DEV)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, **_inputs(case, seed)}
    if kind in ("dropin", "natural", "split"):
        nx, n, batch = case["nx"], case["n"], case["batch"]
        s["plan"] = Plan2D(nx, n, batch) if nx else Plan1D(n, batch)
        s["out"] = torch.empty_like(s["x"])
        s["direction"] = INVERSE if case["inverse"] else FORWARD
        if kind == "split":
            s["plan"].prepare_split()
        if kind == "dropin":  # the order the caller stages its input in
            if nx:
                x = s["x"].index_select(1, _reversal(s["plan"].radices_x, nx))
                s["x"] = x.index_select(2, _reversal(s["plan"].radices_y, n)).contiguous()
            else:
                s["x"] = s["x"].index_select(1, _reversal(s["plan"].radices, n)).contiguous()
    elif kind == "uneven":
        s["plan"] = MultiPlan(_sizes(case))
        s["out"] = torch.empty_like(s["x"])
        s["direction"] = INVERSE if case["inverse"] else FORWARD
    elif kind == "conv":
        s["layer"] = torch_fft.FFTConv1d(case["channels"], case["n"], device=DEV)
        with torch.no_grad():
            s["layer"].weight.copy_(s.pop("h"))
    if case.get("grad"):
        s["x"].requires_grad_(True)
    return s


def run(state):
    case, x = state["case"], state["x"]
    kind = case["kind"]
    if kind in ("fft", "fft32", "rfft"):
        if kind == "fft":
            f = torch_fft.fft_adjoint if case["inverse"] else torch_fft.fft
        elif kind == "fft32":
            f = torch_fft.fft32_adjoint if case["inverse"] else torch_fft.fft32
        else:
            f = torch_fft.rfft
        y = f(x)
        if not case["grad"]:
            return y
        return y, torch.autograd.grad(y, x, state["gy"])[0]
    if kind == "c2r":
        return torch_fft.c2r(x, case["n"])
    if kind == "conv":
        layer = state["layer"]
        if not case["grad"]:
            with torch.no_grad():
                return layer(x)
        y = layer(x)
        return (y, *torch.autograd.grad(y, (x, layer.weight), state["gy"]))
    plan, out, direction = state["plan"], state["out"], state["direction"]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "dropin":
        out.copy_(x)
        plan.exec(out.data_ptr(), direction, stream)
    elif kind == "split":
        plan.exec_split(x.data_ptr(), out.data_ptr(), direction, stream)
    else:
        plan.exec_natural(x.data_ptr(), out.data_ptr(), direction, stream)
    return out


def _cplx(x):
    return x.to(torch.complex128) if x.is_complex() else torch.view_as_complex(x.double().contiguous())


def _dft(z, inverse, dims=(-1,)):
    """Unnormalised transform over the last one or two axes."""
    return torch.fft.ifftn(z, dim=dims, norm="forward") if inverse else torch.fft.fftn(z, dim=dims)


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "uneven":
        z, out, at = _cplx(t["x"]), [], 0
        for n in _sizes(case):
            out.append(_dft(z[at:at + n], case["inverse"]))
            at += n
        return torch.view_as_real(torch.cat(out))
    if kind in ("fft", "dropin", "natural", "split", "fft32"):
        inv = case["inverse"]
        dims = (-2, -1) if case.get("nx") else (-1,)
        real = kind != "fft32"
        y = _dft(_cplx(t["x"]), inv, dims)
        y = torch.view_as_real(y) if real else y
        if not case.get("grad"):
            return y
        g = _dft(_cplx(t["gy"]), not inv, dims)
        return y, torch.view_as_real(g) if real else g
    n = case["n"]
    if kind == "c2r":
        return _hermitian(_cplx(t["x"]), n)
    if kind == "rfft":
        y = torch.view_as_real(torch.fft.rfft(t["x"].double()))
        if not case["grad"]:
            return y
        g = _cplx(t["gy"])
        g[..., 1:-1] *= 0.5
        return y, _hermitian(g, n)
    x, h = _cplx(t["x"]), _cplx(t["h"])
    xs = torch.fft.fft(x)
    y = torch.view_as_real(torch.fft.ifft(xs * h))
    if not case["grad"]:
        return y
    gs = torch.fft.fft(_cplx(t["gy"]))
    gx = torch.view_as_real(torch.fft.ifft(gs * h.conj()))
    gw = torch.view_as_real((xs.conj() * gs).sum(0) / n)
    return y, gx, gw


def _hermitian(z, n):
    """Sum over the Hermitian extension of bins 0..n/2 (n times irfft)."""
    z = z.clone()
    z.imag[..., 0] = 0
    z.imag[..., -1] = 0
    return torch.fft.irfft(z, n=n) * n


def work(case):
    kind = case["kind"]
    if kind == "uneven":
        sizes = _sizes(case)
        return {"bytes": 8.0 * sum(sizes), "flops": sum(5.0 * n * math.log2(n) for n in sizes)}
    n, batch = case["n"], case["batch"]
    passes = 2 if case.get("grad") else 1
    if kind in ("rfft", "c2r"):
        return {"bytes": passes * batch * (2.0 * n + 4.0 * (n // 2 + 1)),
                "flops": passes * batch * 2.5 * n * math.log2(n)}
    if kind == "conv":
        points = float(batch * case["channels"] * n)
        weight = 8.0 * case["channels"] * n  # FP32 spectrum, read; its gradient, written
        return {"bytes": passes * (8.0 * points + weight),
                "flops": passes * (10.0 * points * math.log2(n) + 8.0 * points)}
    points = float(batch * n * (case.get("nx") or 1))
    size = 8.0 if kind in ("fft32", "split") else 4.0
    return {"bytes": passes * 2 * size * points,
            "flops": passes * 5.0 * points * math.log2(n * (case.get("nx") or 1))}
