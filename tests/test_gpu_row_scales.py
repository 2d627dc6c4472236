"""Hermitian rows whose two factors differ in magnitude.

The packed row kernel transforms f + i g as one sequence; the rounding errors of
the smaller factor must stay relative to that factor, row by row, and rows of
other magnitudes, of zeros or of NaN in the same block must not matter.

Bar: relative L2 error of every row <= 1e-12 in FP64, <= 1e-5 in FP32 against
64-bit transforms, the bar that rows of equal magnitude have."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = {"complex128": 1e-12, "complex64": 1e-5}
HERMITIAN = 2

# powers of two that multiply f and g; the products stay representable
SCALES = {"complex128": [(0, 0), (-20, 0), (0, -20), (-40, 0), (0, 40), (-300, 0), (0, -700), (-700, 600),
                         (900, -900), (-500, -400), (500, 400)],
          "complex64": [(0, 0), (-20, 0), (0, -20), (-40, 0), (0, 40), (-60, 0), (0, -90), (-90, 80),
                        (100, -100), (-50, -40), (50, 40), (-120, 110)]}


def _modes(rng, rows, H):
    """Stored modes of real fields with decaying spectra."""
    f = (rng.uniform(-1, 1, (rows, H)) + 1j * rng.uniform(-1, 1, (rows, H))) / np.sqrt(1.0 + np.arange(H))
    f[:, 0] = f[:, 0].real
    return f


def _want(f, g, N):
    H = f.shape[1]
    return np.fft.rfft(np.fft.irfft(f, N) * np.fft.irfft(g, N))[:, :H] * N


def _rows(gpu, f, g, m, q, dtype):
    import torch
    from fftwpp_amd._lib import F32, F64, MULT_REAL_BINARY, check, lib
    rows, H = f.shape
    a, b = (torch.tensor(v, dtype=getattr(torch, dtype), device=gpu) for v in (f, g))
    d = ctypes.c_void_p()
    check(lib().fftwpp_amd_dim_create(ctypes.byref(d), 2 * H - 1, m, q, HERMITIAN))
    try:
        check(lib().fftwpp_amd_conv_rows(d, F64 if dtype == "complex128" else F32, MULT_REAL_BINARY,
                                         a.data_ptr(), b.data_ptr(), rows, H, a.data_ptr(), H,
                                         1.0 / (m * q), None))
        torch.cuda.synchronize()
    finally:
        lib().fftwpp_amd_dim_destroy(d)
    return a.cpu().numpy().astype(np.complex128)


def _errors(h, want):
    """Relative error of each row, free of over- and underflow of the squares."""
    s = np.maximum(np.abs(want).max(axis=1, keepdims=True), 1e-300)
    return np.linalg.norm((h - want) / s, axis=1) / np.linalg.norm(want / s, axis=1)


# (m, H, q): q odd and even, H = m and just above m/2, one residue
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("m,H,q", [(16, 16, 3), (32, 17, 2), (64, 64, 3), (128, 128, 3), (128, 42, 1),
                                   (256, 129, 2), (512, 512, 3), (1024, 1000, 3), (2048, 1025, 2)])
def test_rows(gpu, m, H, q, dtype):
    rows = 523                       # the last block is partly empty
    rng = np.random.default_rng(m + H)
    f, g = _modes(rng, rows, H), _modes(rng, rows, H)
    for i in range(rows):
        sf, sg = SCALES[dtype][i % len(SCALES[dtype])]
        f[i] *= 2.0 ** sf
        g[i] *= 2.0 ** sg
    f[7] = g[8] = f[9] = g[9] = 0.0
    # a factor with one strong mode against a flat one
    f[10], g[10] = f[0] * 1e-6, f[1]
    f[10, 1] = 1.0
    f[11, H // 2] = np.nan
    f, g = (v.astype(dtype).astype(np.complex128) for v in (f, g))
    h = _rows(gpu, f, g, m, q, dtype)
    zero, nan = [7, 8, 9], 11
    assert np.all(h[zero] == 0)
    assert np.isnan(h[nan]).all()
    live = np.array([i for i in range(rows) if i not in zero and i != nan])
    assert _errors(h[live], _want(f[live], g[live], m * q)).max() < TOL[dtype]


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("Hy,my", [(16, 16), (100, 128), (300, 512), (600, 1024)])
def test_plan_and_adjoint(gpu, Hy, my, dtype):
    """A factor 2^-40 on one argument is a factor 2^-40 on the product, and on
    the gradients that the argument enters."""
    import torch
    from fftwpp_amd.torch_conv import DeviceConvolution
    Lx, s = 351, 2.0 ** -40
    dt = getattr(torch, dtype)
    plan = DeviceConvolution((Lx, Hy), kind="hermitian", dtype=dt, M=[528, 3 * my], m=[176, my])
    gen = torch.Generator(device=gpu)
    gen.manual_seed(Hy)
    w, a, b = (plan.symmetrized(torch.randn((Lx, Hy), generator=gen, dtype=dt, device=gpu)) for _ in range(3))

    def close(x, y):
        return (x.to(torch.complex128) - s * y.to(torch.complex128)).norm() <= TOL[dtype] * s * y.norm()
    h = plan(a, b)
    assert close(plan(s * a, b), h) and close(plan(a, s * b), h)
    ga, gb = plan.adjoint(w, a, b)
    ga1, gb1 = plan.adjoint(s * w, a, b)
    assert close(ga1, ga) and close(gb1, gb)
    ga1, _ = plan.adjoint(w, a, s * b)
    assert close(ga1, ga)
