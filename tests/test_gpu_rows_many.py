"""Fused rows of the register engines where several rows share a wave or a
block (short rows in large numbers), with row counts that leave the last block
partly empty, and with row strides so large that one launch's block would
exceed a buffer of 2^31 bytes.

Bar: relative L2 error <= 1e-12 in FP64, <= 1e-5 in FP32 against the oracle."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = {"complex128": 1e-12, "complex64": 1e-5}


def _rnd(rng, shape):
    return rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)


def _plan_run(gpu, f, g, kind, dtype, M, m):
    import torch
    from fftwpp_amd.torch_conv import DeviceConvolution
    dt = getattr(torch, dtype)
    plan = DeviceConvolution(f.shape, kind=kind, dtype=dt, M=M, m=m)
    a, b = (torch.tensor(np.ascontiguousarray(v), dtype=dt, device=gpu) for v in (f, g))
    plan.convolve_(a, b)
    torch.cuda.synchronize()
    return a.cpu().numpy().astype(np.complex128), plan


# y rows of (Hy, m, q): H = m, H just below and just above m/2, q even and odd
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("Hy,my,q", [(16, 16, 4), (9, 16, 3), (32, 32, 3), (33, 64, 3), (63, 64, 4),
                                     (100, 128, 3), (128, 128, 3), (129, 256, 2), (256, 256, 3)])
def test_hermitian_rows(gpu, oracle, Hy, my, q, dtype):
    Lx, mx, qx = 351, 176, 3        # 528 = 33 x 16 rows: some blocks partly empty
    rng = np.random.default_rng(Hy)
    f, g = (oracle.symmetrize_x(_rnd(rng, (Lx, Hy))) for _ in range(2))
    h, plan = _plan_run(gpu, f, g, "hermitian", dtype, [mx * qx, my * q], [mx, my])
    N, m, qq = plan.geometry()
    assert m == (mx, my) and N[0] >= 512
    want = oracle.explicit_hconv(f, g, N)
    assert oracle.rel_l2(h, want) < TOL[dtype]


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("Ly,my,q", [(16, 16, 2), (9, 16, 2), (33, 64, 2), (64, 64, 3), (75, 128, 2),
                                     (128, 128, 2), (500, 512, 2), (1000, 2048, 1)])
def test_complex_rows(gpu, oracle, Ly, my, q, dtype):
    Lx, mx, qx = 300, 174, 3        # 522 rows
    rng = np.random.default_rng(Ly)
    f, g = _rnd(rng, (Lx, Ly)), _rnd(rng, (Lx, Ly))
    h, plan = _plan_run(gpu, f, g, "complex", dtype, [mx * qx, my * q], [mx, my])
    N, m, _ = plan.geometry()
    assert m == (mx, my)
    want = oracle.explicit_conv(f, g, N)
    assert oracle.rel_l2(h, want) < TOL[dtype]


# two residue lanes per row (under 512 rows) and an odd number of passes: every
# lane of the block has to reach the same barriers
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("kind,Ly,my,q", [("complex", 900, 1024, 3), ("complex", 2000, 2048, 3),
                                          ("complex", 4000, 4096, 3), ("complex", 4000, 4096, 2),
                                          ("hermitian", 600, 1024, 5), ("hermitian", 1100, 2048, 5)])
def test_few_rows_odd_passes(gpu, oracle, kind, Ly, my, q, dtype):
    rng = np.random.default_rng(Ly)
    f, g = (_rnd(rng, (201, Ly)) for _ in range(2))
    if kind == "hermitian":
        f, g = oracle.symmetrize_x(f), oracle.symmetrize_x(g)
    h, plan = _plan_run(gpu, f, g, kind, dtype, [402, my * q], [201, my])
    N, m, _ = plan.geometry()
    assert m == (201, my)
    want = (oracle.explicit_hconv if kind == "hermitian" else oracle.explicit_conv)(f, g, N)
    assert oracle.rel_l2(h, want) < TOL[dtype]


@pytest.mark.parametrize("L,m,rows,rs", [(16, 16, 10, 1 << 24), (40, 64, 10, 1 << 24),
                                         (200, 256, 7, 1 << 24), (256, 256, 3, 1 << 27)])
def test_rows_of_huge_stride(gpu, oracle, L, m, rows, rs):
    import torch
    from fftwpp_amd._lib import F64, MULT_BINARY, check, lib
    rng = np.random.default_rng(L)
    f, g = _rnd(rng, (rows, L)), _rnd(rng, (rows, L))
    a, b = (torch.zeros((rows - 1) * rs + L, dtype=torch.complex128, device=gpu) for _ in range(2))
    av, bv = (torch.as_strided(t, (rows, L), (rs, 1)) for t in (a, b))
    av.copy_(torch.tensor(f))
    bv.copy_(torch.tensor(g))
    d = ctypes.c_void_p()
    check(lib().fftwpp_amd_dim_create(ctypes.byref(d), L, m, 2, 0))
    try:
        check(lib().fftwpp_amd_conv_rows(d, F64, MULT_BINARY, a.data_ptr(), b.data_ptr(), rows, rs,
                                         a.data_ptr(), rs, 1.0 / (2 * m), None))
        torch.cuda.synchronize()
        h = av.cpu().numpy()
    finally:
        lib().fftwpp_amd_dim_destroy(d)
    for i in range(rows):
        assert oracle.rel_l2(h[i], oracle.direct_conv(f[i], g[i])) < 1e-12, i


@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("L", [100, 128, 129, 255, 256])
def test_rows_256_repeat(gpu, oracle, L, dtype):
    """Rows of 256 points with two residues, an odd number of them in place:
    every row right, and the same bits each time."""
    import torch
    from fftwpp_amd._lib import F32, F64, MULT_BINARY, check, lib
    rows = 20001
    gen = torch.Generator(device=gpu)
    gen.manual_seed(L)
    f, g = (torch.randn(rows, L, generator=gen, dtype=getattr(torch, dtype), device=gpu) for _ in range(2))
    d = ctypes.c_void_p()
    check(lib().fftwpp_amd_dim_create(ctypes.byref(d), L, 256, 2, 0))
    try:
        out = []
        for _ in range(4):
            h = f.clone()
            torch.cuda.synchronize()
            check(lib().fftwpp_amd_conv_rows(d, F64 if dtype == "complex128" else F32, MULT_BINARY,
                                             h.data_ptr(), g.data_ptr(), rows, L, h.data_ptr(), L,
                                             1.0 / 512, None))
            torch.cuda.synchronize()
            out.append(h)
    finally:
        lib().fftwpp_amd_dim_destroy(d)
    assert all(torch.equal(out[0], o) for o in out[1:])
    z = np.fft.ifft(np.fft.fft(f.cpu().numpy().astype(complex), 512) *
                    np.fft.fft(g.cpu().numpy().astype(complex), 512))[:, :L]
    err = np.linalg.norm(out[0].cpu().numpy() - z, axis=1) / np.linalg.norm(z, axis=1)
    assert err.max() < TOL[dtype]
