"""The first adjoint of a plan may be a captured one, after any execution: it
allocates nothing then.

Bar: every replay equals the eager adjoint of a plan of its own to 1e-13 (FP64)."""
import pytest

pytestmark = pytest.mark.gpu


def test_first_adjoint_under_capture(gpu):
    import torch
    from fftwpp_amd.torch_conv import DeviceConvolution
    shape = (41, 33)
    gen = torch.Generator(device=gpu)
    gen.manual_seed(2)
    w, a, b = (torch.randn(shape, generator=gen, dtype=torch.complex128, device=gpu) for _ in range(3))
    want = DeviceConvolution(shape).adjoint(w, a, b)
    plan = DeviceConvolution(shape)
    plan(a, b)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = plan.adjoint(w, a, b)
    for k in range(3):
        for g in got:
            g.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for x, y in zip(got, want):
            assert (x - y).norm() <= 1e-13 * y.norm()
        # eager work of the same plan between the replays
        eager = plan.adjoint(w, a, b)
        torch.cuda.synchronize()
        for x, y in zip(eager, want):
            assert (x - y).norm() <= 1e-13 * y.norm()
