"""The sizes at which the fully implicit step's kernels change, each side against the other: without a
radial stencil the sweeps and the operator act on every radius alone, so a state of many radii must
agree with its parts."""
import numpy as np
import pytest
import torch

from boltzmann_amd import _lib
from test_gpu_fvm_rounding import _operator

pytestmark = pytest.mark.gpu


def _tables(rng, Nr, Nvt, Nx, nvt, nx):
    """Band tables of both signs with 1 + av dt D_0 >= 1 and couplings of at most half of D_0."""
    def pair(N, nd, sign):
        D = rng.uniform(-0.5, 0.5, (nd, N)) / max(nd - 1, 1)
        D[0] = rng.uniform(1.0, 2.0, N)
        return sign * D
    mu = np.linspace(0.1, 0.95, Nvt // 2)
    return dict(cos_vt=np.append(-mu[::-1], mu), vr=rng.uniform(0.5, 2.0, Nr), wq=rng.uniform(0.5, 1.0, Nvt),
                vt_l2r=pair(Nvt, nvt, -1.0), vt_r2l=pair(Nvt, nvt, 1.0), x_l2r=pair(Nx, nx, 1.0),
                x_r2l=pair(Nx, nx, -1.0), axvr=rng.uniform(0.5, 2.0, Nr), ainv=rng.uniform(0.5, 1.0, Nr))


@pytest.mark.parametrize("Nvt,Nx,nvt", [(16, 128, 4), (8, 260, 2), (8, 500, 5), (24, 200, 3), (6, 70, 4)])
def test_plane_against_sweeps(Nvt, Nx, nvt):
    """256 radii take the plane kernel, 40 of them with planes of more than 1600 cells the sweeps.
    The same formulas, the x scan's in the same order; errors of a chain of contractions stay within
    a few eps of its largest value, 1e-13 here."""
    print(f"case: plane of {Nvt} x {Nx}, nvt={nvt}", flush=True)
    rng = np.random.default_rng(Nx)
    Nr, part = 256, 40
    t = _tables(rng, Nr, Nvt, Nx, nvt, 2)
    b = torch.from_numpy(rng.normal(size=(Nr, Nvt, Nx))).cuda()
    E = torch.from_numpy(rng.normal(size=Nx)).cuda()
    keep = []
    op = _operator(Nr, Nvt, Nx, 2, nvt, 2, keep, **t)
    y = torch.empty_like(b)
    _lib.call("bz_fvm_precond_xvtvrc", op, E, 0.3, b, y)
    for r0 in (0, Nr - part):
        cut = {k: (v[r0:r0 + part] if k in ("vr", "axvr", "ainv") else v) for k, v in t.items()}
        ops = _operator(part, Nvt, Nx, 2, nvt, 2, keep, **cut)
        z = torch.empty((part, Nvt, Nx), dtype=torch.float64, device="cuda")
        _lib.call("bz_fvm_precond_xvtvrc", ops, E, 0.3, b[r0:r0 + part].contiguous(), z)
        got = y[r0:r0 + part]
        assert float((got - z).abs().max()) <= 1e-13 * float(z.abs().max())
        # the product's moment of y, from either route
        w1, w2 = torch.empty_like(b), torch.empty_like(z)
        t1, t2 = torch.empty_like(b), torch.empty_like(z)
        _lib.call("bz_fvm_step_product", op, E, 0.1, 0.3, b, t1, w1, None)
        _lib.call("bz_fvm_step_product", ops, E, 0.1, 0.3, b[r0:r0 + part].contiguous(), t2, w2, None)
        assert torch.equal(t1, y) and torch.equal(t2, z)
        assert float((w1[r0:r0 + part] - w2).abs().max()) <= 1e-12 * float(w2.abs().max())


@pytest.mark.parametrize("nvr,nvt,nx", [(4, 4, 2), (3, 3, 3)])
@pytest.mark.parametrize("Nvt,Nx", [(16, 100), (8, 130)])
def test_ordinates_per_thread(nvr, nvt, nx, Nvt, Nx):
    """The step operator with four, two and one ordinates per thread, by the size of the state: rows of
    a large state against states of its first radii (the last of which have other radial
    neighbours).  The same sums in the same order; the compiler may fuse their products otherwise: a
    few eps of the largest term."""
    rng = np.random.default_rng(Nx)
    Nr = 280
    t = _tables(rng, Nr, Nvt, Nx, nvt, nx)
    t.update(sin_vt=rng.uniform(0.1, 1.0, Nvt), adx=rng.uniform(0.5, 2.0, Nr), loss=rng.uniform(0.1, 0.5, Nr))
    for k, shape in (("dvrL", (nvr, Nr)), ("dvrR", (nvr, Nr)), ("dvtL", (nvt, Nvt)), ("dvtR", (nvt, Nvt)),
                     ("dxL", (nx, Nx)), ("dxR", (nx, Nx))):
        t[k] = rng.uniform(-1.0, 1.0, shape)
    E = torch.from_numpy(rng.normal(size=Nx)).cuda()
    x = torch.from_numpy(rng.normal(size=(Nr, Nvt, Nx))).cuda()
    keep, outs = [], {}
    for part in (Nr, 100, 20):
        waves = part * Nvt * Nx // 64
        assert (waves >= 3200, 800 <= waves < 3200, waves < 800)[(Nr, 100, 20).index(part)]
        cut = {k: (v[:part] if k in ("vr", "axvr", "ainv", "adx", "loss") else v[:, :part] if k in ("dvrL", "dvrR") else v)
               for k, v in t.items()}
        op = _operator(part, Nvt, Nx, nvr, nvt, nx, keep, **cut)
        op.dt_x = 0.3
        y = torch.empty((part, Nvt, Nx), dtype=torch.float64, device="cuda")
        _lib.call("bz_fvm_rhs_mvec", op, E, 0.2, x[:part].contiguous(), y)
        outs[part] = y
    for part in (100, 20):
        n = part - (nvr - 1)
        assert float((outs[part][:n] - outs[Nr][:n]).abs().max()) <= 1e-14 * float(outs[Nr].abs().max())


@pytest.mark.parametrize("nvr,nvt,nx", [(4, 4, 2), (3, 3, 3)])
def test_states_past_32_bit_offsets(nvr, nvt, nx):
    """5.4e8 elements (4.3 GB): the last radii against a state that holds those only; the same kernel
    but for the width of its offsets, so the same bits."""
    Nr, Nvt, Nx, part = 1024, 64, 8300, 12
    assert Nr * Nvt * Nx >= 1 << 29
    rng = np.random.default_rng(nx)
    t = _tables(rng, Nr, Nvt, Nx, nvt, nx)
    t.update(sin_vt=rng.uniform(0.1, 1.0, Nvt), adx=rng.uniform(0.5, 2.0, Nr), loss=rng.uniform(0.1, 0.5, Nr))
    t.pop("ainv")
    for k, shape in (("dvrL", (nvr, Nr)), ("dvrR", (nvr, Nr)), ("dvtL", (nvt, Nvt)), ("dvtR", (nvt, Nvt)),
                     ("dxL", (nx, Nx)), ("dxR", (nx, Nx))):
        t[k] = rng.uniform(-1.0, 1.0, shape)
    E = torch.from_numpy(rng.normal(size=Nx)).cuda()
    gen = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn((Nr, Nvt, Nx), dtype=torch.float64, device="cuda", generator=gen)
    y = torch.empty_like(x)
    keep = []
    op = _operator(Nr, Nvt, Nx, nvr, nvt, nx, keep, **t)
    op.dt_x = 0.3
    _lib.call("bz_fvm_rhs_mvec", op, E, 0.2, x, y)
    cut = {k: (v[-part:] if k in ("vr", "axvr", "adx", "loss") else v[:, -part:] if k in ("dvrL", "dvrR") else v)
           for k, v in t.items()}
    ops = _operator(part, Nvt, Nx, nvr, nvt, nx, keep, **cut)
    ops.dt_x = 0.3
    z = torch.empty((part, Nvt, Nx), dtype=torch.float64, device="cuda")
    _lib.call("bz_fvm_rhs_mvec", ops, E, 0.2, x[-part:].contiguous(), z)
    k = part - (nvr - 1)
    assert torch.equal(y[-k:], z[-k:])
