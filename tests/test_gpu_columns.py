"""Column transforms where their launches differ: 256-point columns in few
tiles (residues dealt to different blocks) and in more tiles than blocks stay
resident, partly filled tiles, real columns over every residue pattern, several
arrays in one launch, and the adjoint's shared transform of the cotangent.

Bar: relative L2 error <= 1e-12 in FP64, <= 1e-5 in FP32 against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = {"complex128": 1e-12, "complex64": 1e-5, "float64": 1e-12, "float32": 1e-5}


def _rnd(rng, shape, real=False):
    u = rng.uniform(-1, 1, shape)
    return u if real else u + 1j * rng.uniform(-1, 1, shape)


def _conv(gpu, f, g, kind, dtype, M=None, m=None):
    import torch
    from fftwpp_amd.torch_conv import DeviceConvolution
    dt = getattr(torch, dtype)
    plan = DeviceConvolution(f.shape, kind=kind, dtype=dt, M=M, m=m)
    a, b = (torch.tensor(np.ascontiguousarray(v), dtype=dt, device=gpu) for v in (f, g))
    out = plan.convolve_out(torch.empty_like(a), a, b)
    torch.cuda.synchronize()
    return out.cpu().numpy(), plan


# x columns of m = 256 (Lx <= 256), q = 1 ... 4; Ly columns: one tile, partly
# filled last tiles, and 125 tiles (63 in FP32)
@pytest.mark.parametrize("kind,dtype", [("complex", "complex128"), ("complex", "complex64"),
                                        ("real", "float64"), ("real", "float32")])
@pytest.mark.parametrize("Lx,Mx,Ly", [(256, 512, 8), (256, 512, 21), (100, 256, 40), (255, 768, 33),
                                      (256, 1024, 19), (130, 512, 1000)])
def test_columns_256(gpu, oracle, Lx, Mx, Ly, kind, dtype):
    rng = np.random.default_rng(Lx + Ly)
    f, g = (_rnd(rng, (Lx, Ly), kind == "real") for _ in range(2))
    h, plan = _conv(gpu, f, g, kind, dtype, M=[Mx, 2 * Ly], m=[256, 0])
    N, m, q = plan.geometry()
    assert m[0] == 256 and N[0] == Mx
    want = oracle.explicit_conv(f, g, N)
    assert oracle.rel_l2(h, want.real if kind == "real" else want) < TOL[dtype]


@pytest.mark.parametrize("kind,dtype", [("complex", "complex128"), ("complex", "complex64"),
                                        ("real", "float64"), ("real", "float32")])
def test_columns_256_many_tiles(gpu, oracle, kind, dtype):
    """About 4000 (FP64) and 2000 (FP32) tiles of columns, the last partly filled."""
    rng = np.random.default_rng(7)
    Lx, Ly, Lz = 200, 71, 449
    f, g = (_rnd(rng, (Lx, Ly, Lz), kind == "real") for _ in range(2))
    h, plan = _conv(gpu, f, g, kind, dtype, M=[512, 142, 898], m=[256, 0, 0])
    want = oracle.explicit_conv(f, g, plan.geometry()[0], workers=8)
    assert oracle.rel_l2(h, want.real if kind == "real" else want) < TOL[dtype]


# few columns: the residues of both arrays are dealt to different blocks
@pytest.mark.parametrize("dtype", ["complex128", "complex64"])
@pytest.mark.parametrize("Lx,mx,qx,Ly", [(20, 16, 5, 9), (100, 128, 2, 17), (300, 512, 2, 24), (600, 512, 3, 40),
                                         (1500, 1024, 3, 16), (3000, 4096, 2, 10)])
def test_few_columns(gpu, oracle, Lx, mx, qx, Ly, dtype):
    rng = np.random.default_rng(Lx)
    f, g = (_rnd(rng, (Lx, Ly)) for _ in range(2))
    h, plan = _conv(gpu, f, g, "complex", dtype, M=[mx * qx, 2 * Ly], m=[mx, 0])
    assert plan.geometry()[1][0] == mx
    assert oracle.rel_l2(h, oracle.explicit_conv(f, g, plan.geometry()[0])) < TOL[dtype]


@pytest.mark.parametrize("kind", ["complex", "hermitian"])
@pytest.mark.parametrize("shape", [(5, 4), (41, 300), (255, 64), (63, 31, 9)])
def test_adjoint_shared(gpu, kind, shape):
    """Both cotangents at once (one transform of the cotangent for 2D plans)
    and each alone agree, and no input changes."""
    import torch
    from fftwpp_amd.torch_conv import DeviceConvolution
    plan = DeviceConvolution(shape, kind=kind)
    g = torch.Generator(device=gpu)
    g.manual_seed(3)
    w, a, b = (torch.randn(shape, generator=g, dtype=torch.complex128, device=gpu) for _ in range(3))
    keep = [t.clone() for t in (w, a, b)]
    ga, gb = plan.adjoint(w, a, b)
    ga1, none = plan.adjoint(w, a, b, need_b=False)
    none2, gb1 = plan.adjoint(w, a, b, need_a=False)
    assert none is None and none2 is None
    for x, y in ((ga, ga1), (gb, gb1)):
        assert (x - y).norm() <= 1e-13 * y.norm()
    assert all(torch.equal(x, y) for x, y in zip(keep, (w, a, b)))


def test_call_keeps_what_it_accepted(gpu):
    """plan(a, b) of an expanded input, as before, and of a tracked one."""
    import torch
    from fftwpp_amd.torch_conv import DeviceConvolution
    plan = DeviceConvolution((6, 5))
    a = torch.randn(5, dtype=torch.complex128, device=gpu).expand(6, 5)
    b = torch.randn(6, 5, dtype=torch.complex128, device=gpu)
    want = plan(a.contiguous(), b)
    assert torch.equal(plan(a, b), want)
    t = a.contiguous().requires_grad_(True)
    assert torch.equal(plan(t, b).detach(), want)


@pytest.mark.parametrize("kind", ["complex", "hermitian"])
def test_call_resolves_lazy_conjugates(gpu, kind):
    """A first factor that is a lazy conjugate is read as its values (both
    factors where the plan symmetrizes copies of them)."""
    import torch
    from fftwpp_amd.torch_conv import DeviceConvolution, convolve
    plan = DeviceConvolution((7, 5), kind=kind)
    a, b = (torch.randn(7, 5, dtype=torch.complex128, device=gpu) for _ in range(2))
    want = plan(a.conj().resolve_conj(), b)
    assert torch.equal(plan(a.conj(), b), want)
    if kind == "hermitian":
        assert torch.equal(plan.symmetrized(a.conj()), plan.symmetrized(a.conj().resolve_conj()))
        ac, bc = a.conj().resolve_conj(), b.conj().resolve_conj()
        assert torch.equal(convolve(a.conj(), b.conj(), plan), convolve(ac, bc, plan))
    else:
        assert torch.equal(convolve(a.conj(), b, plan), want)
