"""Fused multipliers see the rows that exist, and only those: a functor reads a
table of one weight per row (tests/support/fusedmult.hip, RowTable), records the
rows that are bound and counts the products of each.  The table goes on, past
the rows, with entries that no row may touch.  Row counts leave the last block
of each row kernel partly empty.

Bar: every row bound and multiplied once per padded point (the last row, which
empty slots repeat, at least once), no entry past the rows touched, and with unit weights the library's product (relative L2 <= 1e-13
in FP64, 1e-6 in FP32: the same arithmetic, in another compilation)."""
import ctypes
import os

import pytest

pytestmark = pytest.mark.gpu

TESTLIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "support", "libtestmult.so")
GUARD = 512


# (kind, shape, M, m): one row, and 525 = 3 x 175 rows
@pytest.mark.parametrize("double", [True, False])
@pytest.mark.parametrize("kind,shape,M,m", [
    ("complex", (60,), [128], [128]), ("complex", (100,), [256], [128]), ("complex", (200,), [768], [256]),
    ("complex", (350, 9), [525, 32], [175, 16]), ("complex", (350, 75), [525, 256], [175, 128]),
    ("complex", (350, 256), [525, 512], [175, 256]), ("complex", (350, 256), [525, 768], [175, 256]),
    ("complex", (350, 1000), [525, 2048], [175, 1024]), ("centered", (201,), [302], [256]),
    ("hermitian", (100,), [384], [128]), ("hermitian", (349, 16), [525, 48], [175, 16]),
    ("hermitian", (349, 100), [525, 384], [175, 128]), ("hermitian", (349, 256), [525, 768], [175, 256]),
    ("hermitian", (349, 600), [525, 2048], [175, 1024])])
def test_rows_that_exist(gpu, kind, shape, M, m, double):
    import torch
    from fftwpp_amd import _lib
    from fftwpp_amd.torch_conv import DeviceConvolution
    fn = ctypes.CDLL(TESTLIB).fusedmult_table
    fn.argtypes = [ctypes.c_void_p] * 8
    dtype = torch.complex128 if double else torch.complex64
    plan = DeviceConvolution(shape, kind=kind, dtype=dtype, M=M, m=m)
    N, mm, q = plan.geometry()
    assert mm[-1] == m[-1]
    rows = N[0] if len(shape) == 2 else 1
    gen = torch.Generator(device=gpu)
    gen.manual_seed(5)
    a, b = (torch.randn(shape, generator=gen, dtype=dtype, device=gpu) for _ in range(2))
    if kind == "hermitian":
        a, b = plan.symmetrized(a), plan.symmetrized(b)
    w = torch.full((rows + GUARD,), float("nan"), dtype=torch.float64, device=gpu)
    w[:rows] = 1.0
    bound, calls = (torch.zeros(rows + GUARD, dtype=torch.int32, device=gpu) for _ in range(2))
    out, want = torch.empty_like(a), torch.empty_like(a)
    plan.convolve_out(want, a, b)
    torch.cuda.synchronize()
    _lib.check(fn(plan._h, out.data_ptr(), a.data_ptr(), b.data_ptr(), w.data_ptr(), bound.data_ptr(),
                  calls.data_ptr(), None))
    torch.cuda.synchronize()
    assert (bound[:rows] == 1).all() and (bound[rows:] == 0).all()
    assert (calls[:rows - 1] == N[-1]).all() and calls[rows - 1] >= N[-1] and (calls[rows:] == 0).all()
    assert (out - want).norm() <= (1e-13 if double else 1e-6) * want.norm()
