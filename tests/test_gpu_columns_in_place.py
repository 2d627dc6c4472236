"""Forward column transforms in place: a column is read before its residues are
written, also where few columns have their residues dealt to several blocks.

Bar: the same bits as out of place (the same arithmetic on the same words)."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def _forward(d, dtype, f, S, C, nbatch, bsi, F, SF, bso, r0, nres):
    from fftwpp_amd._lib import check, lib
    check(lib().fftwpp_amd_forward_many(d, dtype, f.data_ptr(), S, C, nbatch, bsi, F.data_ptr(), SF, bso,
                                        r0, nres, None))


# 256-point columns in full tiles, other register sizes with L up to 2 m, residues from r0 on
@pytest.mark.parametrize("double", [True, False])
@pytest.mark.parametrize("L,m,q,r0,C,nbatch", [(200, 256, 3, 0, 32, 1), (256, 256, 4, 1, 16, 2), (20, 16, 5, 0, 9, 1),
                                               (100, 64, 4, 0, 70, 1), (600, 512, 3, 0, 24, 2), (1024, 1024, 2, 0, 8, 1),
                                               (3000, 2048, 3, 0, 1, 1), (4096, 4096, 2, 0, 5, 1)])
def test_forward_in_place(gpu, L, m, q, r0, C, nbatch, double):
    import torch
    from fftwpp_amd._lib import F32, F64, check, lib
    dtype = torch.complex128 if double else torch.complex64
    nres = q - r0
    words = max(nres * m, L) * C
    gen = torch.Generator(device=gpu)
    gen.manual_seed(L)
    f = torch.randn((nbatch, words), generator=gen, dtype=dtype, device=gpu)
    F = torch.zeros_like(f)
    torch.cuda.synchronize()
    d = ctypes.c_void_p()
    check(lib().fftwpp_amd_dim_create(ctypes.byref(d), L, m, q, 0))
    try:
        code = F64 if double else F32
        _forward(d, code, f, C, C, nbatch, words, F, C, words, r0, nres)
        _forward(d, code, f, C, C, nbatch, words, f, C, words, r0, nres)
        torch.cuda.synchronize()
    finally:
        lib().fftwpp_amd_dim_destroy(d)
    n = nres * m * C
    assert F[:, :n].abs().max() > 0
    assert torch.equal(f[:, :n], F[:, :n])
