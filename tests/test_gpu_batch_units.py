"""Default work units at the edges of their rules: the lengths where the
sub-FFT size or the number of residues changes, one item and a few hundred
(resident grids, sliced folds), and a single long row, whose output may
replace an input.

Bar: relative L2 error <= 1e-12 in FP64, <= 1e-5 in FP32 against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = [512, 513, 1024, 1025, 2048, 2049, 4096, 4097, 8192, 8193, 16384]


def _pair(L, seed):
    rng = np.random.default_rng(seed)
    return [rng.uniform(-1, 1, L) + 1j * rng.uniform(-1, 1, L) for _ in range(2)]


def _want(oracle, f, g):
    return oracle.explicit_conv(f, g, 1 << (2 * len(f) - 1).bit_length())


@pytest.mark.parametrize("dtype,tol", [("complex128", 1e-12), ("complex64", 1e-5)])
@pytest.mark.parametrize("L", LENGTHS)
def test_default_units(gpu, oracle, L, dtype, tol):
    import torch
    from fftwpp_amd.batch import BatchedConvolution
    for count in (1, 3, 300 if L <= 2049 else 17):
        pairs = [_pair(L, k % 3) for k in range(count)]
        plan = BatchedConvolution([L] * count, dtype=getattr(torch, dtype))
        f, g = (plan.pack([p[k] for p in pairs]) for k in range(2))
        got = plan.unpack(plan(f, g))
        want = [_want(oracle, *p) for p in pairs[:3]]
        assert all(oracle.rel_l2(got[k], want[k % 3]) < tol for k in range(count))


@pytest.mark.parametrize("dtype,tol", [("complex128", 1e-12), ("complex64", 1e-5)])
@pytest.mark.parametrize("shape", [(2049,), (3000,), (4096,), (5, 4000), (4097,), (10000,), (30000,), (3, 5000)])
def test_long_rows(gpu, oracle, shape, dtype, tol):
    import torch
    from fftwpp_amd.torch_conv import DeviceConvolution
    rng = np.random.default_rng(shape[-1])
    f, g = (rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape) for _ in range(2))
    plan = DeviceConvolution(shape, dtype=getattr(torch, dtype))
    a, b = (torch.tensor(v, dtype=plan.dtype, device=gpu) for v in (f, g))
    want = oracle.explicit_conv(f, g, plan.geometry()[0])
    out = plan.convolve_out(torch.empty_like(a), a, b)
    assert oracle.rel_l2(out.cpu().numpy(), want) < tol
    assert torch.equal(plan.convolve_out(b, a, b), out)
