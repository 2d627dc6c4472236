"""The work that programs give this framework, as cases to be timed.

Every case goes through the public Python entry points (DeviceConvolution,
convolve() with its backward, BatchedConvolution, DeviceFFT) on device tensors,
with the plan made once and kept, as a program keeps it.  A case is a dict:

  what      "conv" (one dealiased convolution), "grad" (forward and backward of
            a squared-error loss), "batch" (uneven 1D convolutions) or "fft"
  kind      conv/grad: "complex", "hermitian" or "real"; fft: "c2c", "r2c", "c2r"
  nx ny nz  stored sizes (0: the dimension is absent)
  pad2      conv: 1 pads every dimension to exactly 2 L, 0 takes the default
  double    1: complex128 / float64, 0: complex64 / float32
  sign      fft c2c: the sign of the exponent
  count lo hi   batch: items and the range of their log-uniform lengths
"""
import math
import random

import numpy as np
import torch

from fftwpp_amd.batch import BatchedConvolution
from fftwpp_amd.torch_conv import DeviceConvolution, convolve
from fftwpp_amd.torch_fft import DeviceFFT

DEV = "cuda"


def _conv(name, kind, shape, double=1, pad2=0, what="conv"):
    s = tuple(shape) + (0,) * (3 - len(shape))
    c = {"what": what, "kind": kind, "nx": s[0], "ny": s[1], "nz": s[2], "pad2": pad2, "double": double}
    return dict(c, name=name) if name else c


def _batch(name, count, lo, hi, double=1):
    c = {"what": "batch", "count": count, "lo": lo, "hi": hi, "double": double}
    return dict(c, name=name) if name else c


def _fft(name, kind, shape, double=1, sign=-1):
    s = tuple(shape) + (0,) * (3 - len(shape))
    c = {"what": "fft", "kind": kind, "nx": s[0], "ny": s[1], "nz": s[2], "double": double, "sign": sign}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one short convolution in a loop (filtering, a 1D solver's product): latency
        _conv("conv1d_1024_f64", "complex", (1024,), pad2=1),
        # one long signal of a length nobody chose for the transform
        _conv("conv1d_10000_f32", "complex", (10000,), double=0),
        # image-sized 2D convolution
        _conv("conv2d_1000_f64", "complex", (1000, 1000)),
        # the nonlinear term of a 2D pseudospectral vorticity solver (3/2 rule)
        _conv("herm2d_2047x1024_f64", "hermitian", (2047, 1024)),
        # a training step through that term: value and both gradients
        _conv("herm2d_grad_1023x512_f32", "hermitian", (1023, 512), double=0, what="grad"),
        # one product of a 3D pseudospectral solver of 256 modes a side
        _conv("herm3d_255x255x128_f64", "hermitian", (255, 255, 128)),
        # large 3D convolution, both precisions (the headline workload)
        _conv("conv3d_256_f64", "complex", (256, 256, 256), pad2=1),
        _conv("conv3d_256_f32", "complex", (256, 256, 256), double=0, pad2=1),
        # 3D data of uneven, not power-of-two sides
        _conv("conv3d_100x75x120_f64", "complex", (100, 75, 120)),
        # real 3D data (volume filtering)
        _conv("real3d_256_f64", "real", (256, 256, 256), pad2=1),
        # thousands of uneven 1D signals in one call
        _batch("batch_4096_f64", 4096, 64, 16384),
        # the standalone transform of a 3D field
        _fft("fft3d_256_f64", "c2c", (256, 256, 256)),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _odd(n):
    return n | 1


def _smooth(n):
    """The next length with no prime factor above 7, as programs choose transform lengths."""
    while True:
        r = n
        for p in (2, 3, 5, 7):
            while r % p == 0:
                r //= p
        if r == 1:
            return n
        n += 1


def draw(rng):
    what = rng.choice(["conv1d", "conv2d", "conv3d", "herm2d", "herm3d", "real", "grad", "batch", "fft"])
    double = rng.choice([0, 1])
    pad2 = rng.choice([0, 0, 1])
    if what == "conv1d":
        return _conv(None, "complex", (_log(rng, 64, 16384),), double, pad2)
    if what == "conv2d":
        return _conv(None, "complex", (_log(rng, 32, 1024), _log(rng, 32, 1024)), double, pad2)
    if what == "conv3d":
        return _conv(None, "complex", [rng.randint(32, 256) for _ in range(3)], double, pad2)
    if what == "herm2d":
        return _conv(None, "hermitian", (_odd(_log(rng, 63, 2046)), _log(rng, 32, 1024)), double)
    if what == "herm3d":
        return _conv(None, "hermitian", (_odd(rng.randint(31, 254)), _odd(rng.randint(31, 254)), rng.randint(16, 128)),
                     double)
    if what == "real":
        if rng.random() < 0.4:
            return _conv(None, "real", (_log(rng, 32, 1024), _log(rng, 32, 1024)), double, pad2)
        return _conv(None, "real", [rng.randint(32, 256) for _ in range(3)], double, pad2)
    if what == "grad":
        if rng.random() < 0.5:
            return _conv(None, "complex", (_log(rng, 32, 512), _log(rng, 32, 512)), double, what="grad")
        return _conv(None, "hermitian", (_odd(_log(rng, 63, 1022)), _log(rng, 32, 512)), double, what="grad")
    if what == "batch":
        lo = _log(rng, 16, 256)
        return _batch(None, _log(rng, 256, 4096), lo, _log(rng, 4 * lo, 16384), double)
    kind = rng.choice(["c2c", "c2c", "r2c", "c2r"])
    dims = rng.choice([1, 2, 3])
    if dims == 1:
        n = 2 ** rng.randint(8, 20) if rng.random() < 0.5 else rng.choice([1, 3, 5, 7, 15]) * 2 ** rng.randint(6, 16)
        shape = (n,)
    elif dims == 2:
        shape = [_smooth(_log(rng, 32, 2048)) for _ in range(2)]
    else:
        shape = [_smooth(rng.randint(32, 256)) for _ in range(3)]
    return _fft(None, kind, shape, double, rng.choice([-1, 1]))


def _shape(case):
    return tuple(case[k] for k in ("nx", "ny", "nz") if case[k])


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _uniform(shape, g, real=False):
    """Values uniform in [-1, 1], in 64 bits."""
    if real:
        return 2 * torch.rand(shape, generator=g, dtype=torch.float64, device=DEV) - 1
    return torch.view_as_complex(2 * torch.rand(tuple(shape) + (2,), generator=g, dtype=torch.float64, device=DEV) - 1)


def _mirror(t):
    """The plane t[..., 0] of centred Hermitian data at -k."""
    return torch.flip(t[..., 0], dims=tuple(range(t.dim() - 1)))


def _spectrum(shape, g):
    """Stored modes of a real field: amplitude 1/|k|, random phase, the plane of zero last wavenumber conjugate-symmetric."""
    k2 = 0
    for a, n in enumerate(shape):
        k = torch.arange(n, dtype=torch.float64, device=DEV) - (0 if a == len(shape) - 1 else n // 2)
        k2 = k2 + (k * k).reshape([n if b == a else 1 for b in range(len(shape))])
    phase = 2 * math.pi * torch.rand(shape, generator=g, dtype=torch.float64, device=DEV)
    t = torch.polar(k2.clamp(min=1.0).rsqrt(), phase)
    t[..., 0] = 0.5 * (t[..., 0] + _mirror(t).conj())
    return t


def _inputs(case, seed):
    """The case's inputs in 64 bits: a and b, and a target for "grad"."""
    g, shape = _gen(seed), _shape(case)
    n = 3 if case["what"] == "grad" else 2
    if case["kind"] == "hermitian":
        return [_spectrum(shape, g) for _ in range(n)]
    return [_uniform(shape, g, case["kind"] == "real") for _ in range(n)]


def _cplx(case):
    return torch.complex128 if case["double"] else torch.complex64


def _real(case):
    return torch.float64 if case["double"] else torch.float32


def _lengths(case):
    """Item lengths: the same for every seed, as a program that convolves new data of one layout meets them."""
    r = random.Random(1000003 * case["count"] + 8191 * case["lo"] + case["hi"])
    return [_log(r, case["lo"], case["hi"]) for _ in range(case["count"])]


def prepare(case, seed):
    if case["what"] == "batch":
        plan = BatchedConvolution(_lengths(case), dtype=_cplx(case))
        g = _gen(seed)
        f, h = (_uniform((plan.size,), g).to(_cplx(case)) for _ in range(2))
        return {"what": "batch", "plan": plan, "f": f, "g": h, "out": torch.empty_like(f)}
    if case["what"] == "fft":
        shape, kind = _shape(case), case["kind"]
        x = _fft_input(case, seed)
        half = shape[:-1] + (shape[-1] // 2 + 1,)
        x = x.to(_real(case) if kind == "r2c" else _cplx(case))
        if kind == "c2r":
            out = torch.empty(shape, dtype=_real(case), device=DEV)
        else:
            out = torch.empty(half if kind == "r2c" else shape, dtype=_cplx(case), device=DEV)
        return {"what": "fft", "plan": DeviceFFT(shape, case["sign"], kind, _real(case)), "x": x, "out": out}
    shape = _shape(case)
    dtype = _real(case) if case["kind"] == "real" else _cplx(case)
    M = [2 * n for n in shape] if case["pad2"] else None
    t = [v.to(dtype) for v in _inputs(case, seed)]
    state = {"what": case["what"], "plan": DeviceConvolution(shape, kind=case["kind"], dtype=dtype, M=M), "a": t[0], "b": t[1]}
    if case["what"] == "grad":
        state["t"] = t[2]
        for v in t[:2]:
            v.requires_grad_(True)
    else:
        state["out"] = torch.empty_like(t[0])
    return state


def run(state):
    plan = state["plan"]
    if state["what"] == "batch":
        return plan(state["f"], state["g"], state["out"])
    if state["what"] == "fft":
        return plan(state["x"], state["out"])
    if state["what"] == "grad":
        h = convolve(state["a"], state["b"], plan)
        d = h - state["t"]
        loss = torch.view_as_real(d).square().sum()
        ga, gb = torch.autograd.grad(loss, (state["a"], state["b"]))
        return {"h": h, "loss": loss, "ga": ga, "gb": gb}
    return plan.convolve_out(state["out"], state["a"], state["b"])


def work(case):
    """Bytes: each input read and each output written once.  Flops: 5 N log2 N per transform of the padded length."""
    E = 16 if case["double"] else 8
    if case["what"] == "batch":
        L = _lengths(case)
        return {"bytes": 3 * E * sum(L), "flops": sum(15 * 2 * n * math.log2(2 * n) for n in L)}
    shape = _shape(case)
    n = math.prod(shape)
    if case["what"] == "fft":
        half = math.prod(shape[:-1]) * (shape[-1] // 2 + 1)
        full = 5 * n * math.log2(max(2, n))
        return {"bytes": 2 * E * n, "flops": full} if case["kind"] == "c2c" else {"bytes": E // 2 * n + E * half, "flops": full / 2}
    if case["kind"] == "hermitian":
        N = math.prod(1.5 * s for s in shape[:-1]) * 3 * shape[-1] / 2
        arrays, E1 = 3, E
    else:
        N = math.prod(2 * s for s in shape)
        arrays, E1 = 3, E
        if case["kind"] == "real":
            N, E1 = N / 2, E // 2
    flops = 3 * 5 * N * math.log2(max(2.0, N))
    if case["what"] == "grad":
        # forward (a, b -> h), the loss (h, target), backward (its cotangent, a, b -> two gradients)
        return {"bytes": (3 + 2 + 5) * E1 * n, "flops": 8 * 5 * N * math.log2(max(2.0, N))}
    return {"bytes": arrays * E1 * n, "flops": flops}


# ---- the same outputs from torch and numpy in 64 bits


def _pow2(n):
    return 1 << (n - 1).bit_length()


def _linear(a, b):
    """The terms of the linear convolution of a and b that the convolution keeps: as many as the inputs have."""
    dims = tuple(range(a.dim()))
    size = [_pow2(2 * n - 1) for n in a.shape]
    A, B = (torch.fft.fftn(v.to(torch.complex128), s=size, dim=dims) for v in (a, b))
    return torch.fft.ifftn(A * B, dim=dims)[tuple(slice(0, n) for n in a.shape)]


def _symmetric(t):
    """t with its plane of zero last wavenumber made conjugate-symmetric from the modes after the origin."""
    p = t[..., 0]
    q = p.reshape(-1)
    mid = q.numel() // 2
    up = q[mid + 1:]
    q = torch.cat([torch.flip(up, (0,)).conj(), q[mid:mid + 1].real.to(q.dtype), up])
    return torch.cat([q.reshape(p.shape).unsqueeze(-1), t[..., 1:]], dim=-1)


def _hermitian(a, b):
    """Stored modes of the product of two real fields given by their stored modes."""
    shape = a.shape
    full = [*shape[:-1], 2 * shape[-1] - 1]
    # wrapped modes do not reach the stored ones from 3/2 of the length on
    size = [_pow2(3 * ((n + 1) // 2)) for n in full]
    spectra = []
    for v in (a, b):
        neg = torch.flip(v[..., 1:], dims=tuple(range(v.dim()))).conj()
        spectra.append(torch.fft.fftn(torch.cat([neg, v], dim=-1), s=size))
    h = torch.fft.ifftn(spectra[0] * spectra[1])
    # index 0 of a side of n modes is wavenumber -(n // 2), so the product's origin is at 2 (n // 2)
    for axis, n in enumerate(full):
        c = n // 2
        count = shape[-1] if axis == len(full) - 1 else n
        first = 2 * c if axis == len(full) - 1 else c
        idx = (first + torch.arange(count, device=h.device)) % size[axis]
        h = h.index_select(axis, idx)
    return h


def _fft_input(case, seed):
    """Input of a transform; that of c2r is the spectrum of a real field."""
    shape, g = _shape(case), _gen(seed)
    if case["kind"] == "c2c":
        return _uniform(shape, g)
    x = _uniform(shape, g, True)
    if case["kind"] == "r2c":
        return x
    y = np.fft.rfftn(x.cpu().numpy()) / math.sqrt(math.prod(shape))
    return torch.as_tensor(y, device=DEV)


def exact(case, seed):
    if case["what"] == "batch":
        L, g = _lengths(case), _gen(seed)
        off = np.concatenate([[0], np.cumsum(L)])
        f, h = (_uniform((int(off[-1]),), g).to(_cplx(case)).to(torch.complex128) for _ in range(2))
        out = torch.empty_like(f)
        groups = {}
        for i, n in enumerate(L):
            groups.setdefault(_pow2(2 * n - 1), []).append(i)
        for N, items in groups.items():
            for k in range(0, len(items), 256):
                part = items[k:k + 256]
                A = torch.zeros((2, len(part), N), dtype=torch.complex128, device=DEV)
                for j, i in enumerate(part):
                    A[0, j, :L[i]] = f[off[i]:off[i + 1]]
                    A[1, j, :L[i]] = h[off[i]:off[i + 1]]
                A = torch.fft.fft(A)
                y = torch.fft.ifft(A[0] * A[1])
                for j, i in enumerate(part):
                    out[off[i]:off[i + 1]] = y[j, :L[i]]
        return out
    if case["what"] == "fft":
        x = _fft_input(case, seed)
        x = x.to(_real(case) if case["kind"] == "r2c" else _cplx(case)).cpu().numpy()
        n = math.prod(_shape(case))
        if case["kind"] == "r2c":
            return np.fft.rfftn(x.astype(np.float64))
        x = x.astype(np.complex128)
        if case["kind"] == "c2r":
            return np.fft.irfftn(x, s=_shape(case), axes=range(len(_shape(case)))) * n
        return np.fft.fftn(x) if case["sign"] < 0 else np.fft.ifftn(x) * n
    wide = torch.float64 if case["kind"] == "real" else torch.complex128
    narrow = _real(case) if case["kind"] == "real" else _cplx(case)
    t = [v.to(narrow).to(wide) for v in _inputs(case, seed)]
    herm = case["kind"] == "hermitian"
    if case["what"] == "conv":
        # inputs rounded to 32 bits stay conjugate-symmetric, as negation is exact
        h = _hermitian(t[0], t[1]) if herm else _linear(t[0], t[1])
        return h.real if case["kind"] == "real" else h
    a, b = (v.requires_grad_(True) for v in t[:2])
    h = _hermitian(_symmetric(a), _symmetric(b)) if herm else _linear(a, b)
    loss = torch.view_as_real(h - t[2]).square().sum()
    ga, gb = torch.autograd.grad(loss, (a, b))
    return {"h": h.detach(), "loss": loss.detach(), "ga": ga, "gb": gb}
