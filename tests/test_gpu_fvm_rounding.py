"""Rounding of the fully implicit step's kernels against the same formulas evaluated once per element
with fused products, both measured against 64-bit significands on the host."""
import numpy as np
import pytest
import torch

from boltzmann_amd import _lib
from boltzmann_amd.bte_1d3v_solver import column_bands, upwinded_dx

pytestmark = pytest.mark.gpu
LD = np.longdouble


def _fma(a, b, c):
    return (LD(a) * LD(b) + LD(c)).astype(np.float64)


def _operator(Nr, Nvt, Nx, nvr, nvt, nx, keep, **tables):
    op = _lib.Fvm1d3v()
    op.Nr, op.Nvt, op.Nx, op.nvr, op.nvt, op.nx = Nr, Nvt, Nx, nvr, nvt, nx
    z = np.zeros
    t = dict(cos_vt=z(Nvt), sin_vt=z(Nvt), vr=np.ones(Nr), wq=z(Nvt), loss=z(Nr), g_ptr=z(Nr + 1, np.int32),
             g_col=z(1, np.int32), g_val=z(1), dvrL=z((nvr, Nr)), dvrR=z((nvr, Nr)), dvtL=z((nvt, Nvt)),
             dvtR=z((nvt, Nvt)), dxL=z((nx, Nx)), dxR=z((nx, Nx)), adx=z(Nr), vr_l2r=z((nvr, Nr)), vr_r2l=z((nvr, Nr)),
             vt_l2r=z((nvt, Nvt)), vt_r2l=z((nvt, Nvt)), x_l2r=z((nx, Nx)), x_r2l=z((nx, Nx)), axvr=z(Nr),
             ainv=np.ones(Nr), H=z((Nr, Nr)), h_lo=z(Nr, np.int32), work=z(2 * Nr * Nx))
    t.update(tables)
    for k, v in t.items():
        keep.append(torch.from_numpy(np.ascontiguousarray(v)).cuda())
        setattr(op, k, keep[-1].data_ptr())
    op.dt_x, op.tau_n0np0, op.tau, op.eq, op.eaE = 0.0, 0.0, 1.0, 1.0, 1.0
    return op


@pytest.mark.parametrize("Nr,nvr", [(671, 4), (250, 3), (800, 2)])
def test_radial_scan(Nr, nvr):
    """The preconditioner reduced to its radial sweep.  In segments it evaluates the same formula from
    states that are re-associated at rounding level, which contraction damps (dt av D_0 at most one
    here): the 2-norm of its error is that of the sequential sweep to within a few per cent (over
    3e5 values it is a fixed number; a rounding more per position adds 20 %)."""
    Nvt, Nx, dt = 8, 96, 0.01
    print(f"case: radial scan Nr={Nr} nvr={nvr}", flush=True)
    rng = np.random.default_rng(Nr)
    vr = np.linspace(0.02, 6.0, Nr)
    D = {}
    for key, dr in (("L", "L"), ("R", "R")):
        M = upwinded_dx(vr, nvr, dr)
        M[0 if dr == "L" else -1] = 0.0
        D[key] = np.asarray(column_bands(M, nvr, dr == "L"))
    half = rng.uniform(0.2, 1.0, Nvt // 2)
    cos = np.append(-half, half[::-1])
    E = rng.normal(size=Nx) * np.where(np.arange(Nx) % 2 == 0, 0.05, 0.5)
    keep = []
    op = _operator(Nr, Nvt, Nx, nvr, 2, 2, keep, cos_vt=cos, vr_l2r=D["L"], vr_r2l=D["R"])
    b = rng.normal(size=(Nr, Nvt, Nx))
    out = torch.empty(b.shape, dtype=torch.float64, device="cuda")
    _lib.call("bz_fvm_precond_xvtvrc", op, torch.from_numpy(E).cuda(), dt, torch.from_numpy(b).cuda(), out)
    got = out.cpu().numpy()
    av = -(cos[:, None] * E[None])
    exact, plain = np.zeros(b.shape, LD), np.zeros(b.shape)
    for fwd, key in ((True, "L"), (False, "R")):
        m = (av >= 0) == fwd
        a = av[m]
        ye = [np.zeros(a.size, LD)] * nvr
        yp = [np.zeros(a.size)] * nvr
        for p in range(Nr):
            c = p if fwd else Nr - 1 - p
            dd = [D[key][k, min(max(c - k if fwd else c + k, 0), Nr - 1)] for k in range(nvr)]
            se, sp = np.zeros(a.size, LD), np.zeros(a.size)
            for k in range(nvr - 1, 0, -1):
                se = se + LD(dd[k]) * ye[k - 1]
                sp = _fma(dd[k], yp[k - 1], sp)
            ve = (LD(1) * b[c][m] - LD(dt) * a * se) / (1 + LD(dt) * a * LD(dd[0]))
            vp = _fma(-sp, dt * a, b[c][m]) * (1.0 / _fma(a * dt, dd[0], np.ones(a.size)))
            ye, yp = [ve] + ye[:-1], [vp] + yp[:-1]
            exact[c][m], plain[c][m] = ve, vp
    inner = np.ones(b.shape, bool)                       # the x sweep, of zero speed, zeroes its first point
    inner[:, :, 0] = False
    err = lambda x: float(np.linalg.norm(((x - exact) * inner).astype(np.float64)))
    assert err(plain) > 0
    assert err(got) <= 1.08 * err(plain)


@pytest.mark.parametrize("nvr,nvt,nx,Nvt", [(4, 4, 2, 16), (3, 3, 3, 12), (4, 4, 2, 6), (2, 2, 2, 8)])
def test_angular_coefficient(nvr, nvt, nx, Nvt):
    """The step operator reduced to x + (sin / vr) x at x = 1 (one angular weight of one, E = 1): with
    the quotient between 2^20 and 2^21 the sum is exact, so the coefficient is the quotient itself.
    The widths of both fixed stencils, four, two and one ordinates per thread, and the general form."""
    Nr, Nx = 40, 5
    rng = np.random.default_rng(nvr * Nvt)
    sin, vr = rng.uniform(0.75, 1.0, Nvt), 2.0 ** -20 * rng.uniform(0.5, 0.75, Nr)
    Dt = np.zeros((nvt, Nvt))
    Dt[0] = 1.0
    keep = []
    op = _operator(Nr, Nvt, Nx, nvr, nvt, nx, keep, sin_vt=sin, vr=vr, dvtL=Dt, dvtR=Dt)
    x = torch.ones((Nr, Nvt, Nx), dtype=torch.float64, device="cuda")
    y = torch.empty_like(x)
    _lib.call("bz_fvm_rhs_mvec", op, torch.ones(Nx, dtype=torch.float64, device="cuda"), 1.0, x, y)
    q = sin[None] / vr[:, None]
    assert q.min() >= 2.0 ** 20 and q.max() < 2.0 ** 21
    # the velocity term is zero at the inflow points of either half range
    np.testing.assert_array_equal(y.cpu().numpy()[:, :, 1:-1] - 1.0, np.repeat(q[:, :, None], Nx - 2, axis=2))
