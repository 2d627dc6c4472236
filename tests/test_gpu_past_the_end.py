"""Words past the end of an item or a row do not enter it: the items of a batch
between items of NaN, and rows of 256 points whose strides leave NaN between
them, last words of the arrays included.

Bar: relative L2 error <= 1e-12 in FP64, <= 1e-5 in FP32 against 64-bit
transforms."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = {"complex128": 1e-12, "complex64": 1e-5}


def _want(f, g):
    n = f.shape[-1]
    N = 1 << (2 * n - 1).bit_length()
    return np.fft.ifft(np.fft.fft(f, N) * np.fft.fft(g, N))[..., :n]


def _rel(h, want):
    return np.linalg.norm(h - want) / np.linalg.norm(want)


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("L", [300, 513, 1025, 2049, 2050, 4099, 6145, 9000])
def test_items_between_nan(gpu, L, dtype):
    import torch
    from fftwpp_amd.batch import BatchedConvolution
    dt = getattr(torch, dtype)
    plan = BatchedConvolution([L] * 7, dtype=dt)
    rng = np.random.default_rng(L)
    x = rng.uniform(-1, 1, (2, 7, L, 2)) @ np.array([1, 1j])
    x[:, 0::2] = np.nan
    # every second item is NaN; the arrays end inside larger ones of NaN
    f, g, out = (torch.full((plan.size + 8192,), float("nan"), dtype=dt, device=gpu)[:plan.size] for _ in range(3))
    for t, v in ((f, x[0]), (g, x[1])):
        t.copy_(plan.pack(list(v)))
    h = [t.cpu().numpy() if hasattr(t, "cpu") else np.asarray(t) for t in plan.unpack(plan(f, g, out))]
    for i in range(1, 7, 2):
        assert _rel(h[i], _want(x[0, i], x[1, i])) < TOL[dtype]
    assert all(np.isnan(h[i]).all() for i in range(0, 7, 2))


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("L,rs", [(1, 3), (17, 17), (129, 200), (200, 256), (255, 300), (256, 260)])
def test_rows_between_nan(gpu, L, rs, dtype):
    import torch
    from fftwpp_amd._lib import F32, F64, MULT_BINARY, check, lib
    rows = 37
    rng = np.random.default_rng(L)
    f, g = (rng.uniform(-1, 1, (rows, L)) + 1j * rng.uniform(-1, 1, (rows, L)) for _ in range(2))
    f[4::5] = np.nan
    a, b = (torch.full((rows * rs + 4096,), float("nan"), dtype=getattr(torch, dtype), device=gpu) for _ in range(2))
    av, bv = (torch.as_strided(t, (rows, L), (rs, 1)) for t in (a, b))
    av.copy_(torch.tensor(f))
    bv.copy_(torch.tensor(g))
    keep = a.clone()
    torch.as_strided(keep, (rows, L), (rs, 1)).fill_(0)
    d = ctypes.c_void_p()
    check(lib().fftwpp_amd_dim_create(ctypes.byref(d), L, 256, 2, 0))
    try:
        check(lib().fftwpp_amd_conv_rows(d, F64 if dtype == "complex128" else F32, MULT_BINARY, a.data_ptr(),
                                         b.data_ptr(), rows, rs, a.data_ptr(), rs, 1.0 / 512, None))
        torch.cuda.synchronize()
    finally:
        lib().fftwpp_amd_dim_destroy(d)
    h = av.cpu().numpy()
    for i in range(rows):
        if i % 5 == 4:
            assert np.isnan(h[i]).all()
        else:
            assert _rel(h[i], _want(f[i], g[i])) < TOL[dtype]
    # nothing stored between the rows
    av.fill_(0)
    assert torch.equal(torch.view_as_real(a).isnan(), torch.view_as_real(keep).isnan())
