"""The fused preconditioner and step product of bz_fvm.hip against the oracle: the plane kernel (its
x scan at two, four and eight points per lane, every angular stencil) and the sweeps it does not
take (planes past its LDS, three-point x stencils), the step operator's groups of four
ordinates where they do not divide, and the moment shared with the step operator.  Tolerances as for the same products elsewhere:
1e-12 of the largest entry for the preconditioner (dense solves in the oracle), 1e-11 for the step
operator applied to it (its radial differences amplify by about ten)."""
import numpy as np
import pytest
import torch

from test_gpu_fvm1d3v import _field, _pair, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [dict(Np=64), dict(Np=65, pvt=1), dict(Np=130, pvt=2), dict(Np=260, pvt=4, Nvt=10),
                                dict(Np=9, px=2), dict(Nr=5, Nvt=32, Np=251),             # past the LDS of a plane
                                dict(Nvt=10, Np=7), dict(Nvt=14, Np=129),                  # ordinates in uneven groups
                                dict(Nr=27, spline_qpts=5, Np=5), dict(Nr=27, spline_qpts=5, Np=5, pvr=1)])
def test_product_and_preconditioner(kw):
    from boltzmann_amd import _lib
    S, O = _pair(**kw)
    dt = 2e-3
    S.init(dt, 0.8, 0.9)
    O.init(dt, 0.8, 0.9)
    rng = np.random.default_rng(7)
    b = rng.normal(size=(O.dof_v, O.Nx))
    E = _field(O.xp)
    want = O.step_op_split(E, b, dt, alpha=0.6)
    v = torch.from_numpy(b).cuda().reshape(-1)
    t, w = torch.empty_like(v), torch.empty_like(v)
    Ed = S._field(E)
    _lib.call("bz_fvm_step_product", S._op, Ed, dt, 0.6 * dt, v, t, w, None)
    assert _rel(t.reshape(b.shape), want) < 1e-12
    assert torch.equal(t, S.step_op_split(Ed, v, None, 0.0, dt, alpha=0.6).reshape(-1))
    assert _rel(w, O.rhs_mvec(E, want, dt)) < 1e-11
    flag = torch.ones(1, dtype=torch.int32, device="cuda")
    t2, w2 = torch.full_like(t, 3.0), torch.full_like(w, 4.0)
    _lib.call("bz_fvm_step_product", S._op, Ed, dt, 0.6 * dt, v, t2, w2, flag)
    assert bool((t2 == 3.0).all()) and bool((w2 == 4.0).all())
