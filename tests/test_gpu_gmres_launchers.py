"""DeviceGMRES with launchers (src, dst): the same system as with launchers that also take the stop
flag, eagerly and from captured graphs, over several cycles with a last chunk of fewer steps."""
import pytest
import torch

from boltzmann_amd import _lib
from boltzmann_amd.krylov import DeviceGMRES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flag", [False, True])
@pytest.mark.parametrize("use_graph", [False, True])
def test_two_and_three_arguments(flag, use_graph):
    """Both products by this library's kernels, which may be captured.  The solver's own residual
    test bounds the solution: the host's residual differs by rounding, n eps |A| |x|."""
    n, restart = 300, 6
    print(f"case: flag={flag} graph={use_graph}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(3)
    f64 = dict(dtype=torch.float64, device="cuda")
    A = torch.eye(n, **f64) + 0.5 / n ** 0.5 * torch.randn((n, n), generator=gen, **f64)
    P = 0.5 * torch.eye(n, **f64)
    matvec = lambda src, dst: _lib.call("bz_dgemm_nn", A, n, n, src, 1, dst)
    precond = lambda src, dst: _lib.call("bz_dgemm_nn", P, n, n, src, 1, dst)
    if flag:
        mv, pc = lambda src, dst, done: matvec(src, dst), lambda src, dst, done: precond(src, dst)
    else:
        mv, pc = matvec, precond
    s = DeviceGMRES(n, restart, torch.device("cuda"), mv, pc, use_graph=use_graph)
    for rep, tol in enumerate((1e-8, 1e-5, 1e-9)):
        b = torch.randn(n, generator=gen, **f64)
        x0 = None if rep != 1 else torch.randn(n, generator=gen, **f64)
        seen = []
        x, k = s.solve(b, 0.0, tol, 50, x0=x0, callback=seen.append)
        r = torch.linalg.vector_norm(A.cpu() @ x.cpu() - b.cpu()) / torch.linalg.vector_norm(b.cpu())
        assert float(r) < 1.01 * tol and seen[-1] < tol
        assert len(seen) >= 2 and restart < k <= restart * len(seen)


@pytest.mark.parametrize("use_graph", [False, True])
def test_no_callback_for_a_converged_start(use_graph):
    """One call per cycle that was run: none where |b - A P x0| is below the tolerance."""
    n = 40
    f64 = dict(dtype=torch.float64, device="cuda")
    A = 2.0 * torch.eye(n, **f64)
    P = torch.eye(n, **f64)
    s = DeviceGMRES(n, 3, torch.device("cuda"), lambda a, b: _lib.call("bz_dgemm_nn", A, n, n, a, 1, b),
                    lambda a, b: _lib.call("bz_dgemm_nn", P, n, n, a, 1, b), use_graph=use_graph)
    b = torch.arange(1.0, n + 1, **f64)
    seen = []
    for x0, calls, steps in ((None, 1, 1), (0.5 * b, 0, 0), (b, 1, 1), (0.5 * b, 0, 0)):
        del seen[:]
        x, k = s.solve(b, 0.0, 1e-12, 5, x0=x0, callback=seen.append)
        assert (len(seen), k) == (calls, steps)
        assert torch.equal(x, 0.5 * b) or float((x - 0.5 * b).abs().max()) < 1e-12 * n
    x, k = s.solve(0.0 * b, 1e-3, 0.0, 5, callback=seen.append)
    assert k == 0 and not bool(x.any()) and len(seen) == 0


@pytest.mark.parametrize("nx,nbins", [(1023, 1), (1024, 1), (1000, 30), (2000, 256), (4096, 256)])
def test_points_grouped_by_several_workgroups(nx, nbins):
    """Whole numbers: starts, counts and a stable order, with points in every bin, the last included."""
    gen = torch.Generator(device="cuda").manual_seed(nx)
    b = torch.randint(0, nbins, (nx,), generator=gen, dtype=torch.int32, device="cuda")
    b[-1] = nbins - 1
    out = [torch.full((k,), -1, dtype=torch.int32, device="cuda") for k in (nbins, nbins, nx)]
    _lib.call("bz_group_bins", b, nx, nbins, *out)
    count = torch.bincount(b.cpu().long(), minlength=nbins)
    assert torch.equal(out[1].cpu().long(), count)
    assert torch.equal(out[0].cpu().long(), count.cumsum(0) - count)
    assert torch.equal(out[2].cpu().long(), torch.argsort(b.cpu(), stable=True))
