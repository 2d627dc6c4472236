"""Untuned batches on both sides of the rules that depend on the number of items:
two residues of 512 or one of 1024 (FP64), both residues of an item in one unit
or each in its own (FP64 m = 2048, FP32 m = 4096), resident grids.

Bar: relative L2 error <= 1e-12 in FP64, <= 1e-5 in FP32 against 64-bit
transforms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("double,L,count,mq", [
    (True, 257, 4095, (1024, 1)), (True, 257, 4096, (512, 2)), (True, 512, 4100, (512, 2)), (True, 513, 4096, (2048, 1)),
    (True, 1025, 255, (2048, 2)), (True, 2048, 257, (2048, 2)), (False, 2049, 100, (4096, 2)),
    (False, 4096, 511, (4096, 2)), (False, 2500, 513, (4096, 2)), (False, 600, 1500, (2048, 1))])
def test_counts(gpu, double, L, count, mq):
    import torch
    from fftwpp_amd.batch import BatchedConvolution
    dtype = torch.complex128 if double else torch.complex64
    plan = BatchedConvolution([L] * count, dtype=dtype)
    assert plan.geometry(0)[:2] == mq
    gen = torch.Generator(device=gpu)
    gen.manual_seed(L)
    f, g = (torch.randn(plan.size, generator=gen, dtype=dtype, device=gpu) for _ in range(2))
    h = plan(f, g).cpu().numpy().reshape(count, L).astype(np.complex128)
    a, b = (t.cpu().numpy().reshape(count, L).astype(np.complex128) for t in (f, g))
    N = 1 << (2 * L - 1).bit_length()
    err = []
    for i in range(0, count, 64):
        s = slice(i, i + 64)
        z = np.fft.ifft(np.fft.fft(a[s], N) * np.fft.fft(b[s], N))[:, :L]
        err.append((np.linalg.norm(h[s] - z, axis=1) / np.linalg.norm(z, axis=1)).max())
    assert max(err) < (1e-12 if double else 1e-5)
