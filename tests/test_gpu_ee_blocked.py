"""The e-e entry points on tables planned without the e-e pattern (the blocked elimination's): the
checks, and tolerances, of test_gpu_ee at lmax = 1, whose pattern holds the whole e-e operator, and the
preconditioner alone at more windows and tile counts."""
import numpy as np
import pytest
import torch

import test_gpu_ee as ee
from helpers import instance_params, oracle_batched, product_grid, product_xsecs
from oracle import ee as eeo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def setup():
    from boltzmann_amd.bte_ee import EEOperator
    from boltzmann_amd.solver0d import Batched0D
    print("case: e-e on tables without its pattern, Nr=24 lmax=1", flush=True)
    ops, g, procs = oracle_batched(24, 1)
    vg = product_grid(g)
    s = Batched0D(vg, product_xsecs())
    assert s.tables.struct.nslots % 64 != 0
    hl, gl = eeo.rosenbluth_ops(g, ops.Minv)
    A, Bt = eeo.cc_tensors(g)
    return ops, g, s, EEOperator(vg, s), hl, gl, A, Bt


def test_newton_krylov_pieces(setup):
    ee.test_newton_krylov_pieces(setup)


def test_steady_state(setup):
    ee.test_steady_state_with_ee(setup)


@pytest.mark.parametrize("Nr,lmax,nproc,B", [(25, 2, 1, 3), (130, 2, 3, 4), (41, 4, 3, 3), (200, 1, 3, 2), (230, 2, 3, 2)])
def test_preconditioner(Nr, lmax, nproc, B):
    """z = P v solves P (M^-1 K z - mu z) = v for v in u-perp, at the Maxwellian without e-e; the bound
    is the one of test_newton_krylov_pieces.  Both forms of tables, an inactive instance left alone."""
    from boltzmann_amd import _lib
    from boltzmann_amd.bte_ee import _NKWork
    from boltzmann_amd.solver0d import Batched0D
    print(f"case: preconditioner Nr={Nr} lmax={lmax} nproc={nproc} B={B}", flush=True)
    ops, g, procs = oracle_batched(Nr, lmax)
    vg = product_grid(g)
    prm = instance_params(B, seed=Nr)
    n0, Tg, E, ns = (ee._d(prm[k]) for k in ("n0", "Tg", "E", "ns_by_n0"))
    ns = ns[:nproc].contiguous()
    n, npr, nh = vg.n, vg.npr, vg.num_sh
    rng = np.random.default_rng(3)
    for pattern in (False, True):
        s = Batched0D(vg, product_xsecs()[:nproc], growth="collisions", ee_pattern=pattern)
        assert (s.tables.struct.nslots % 64 == 0) == pattern
        x = s.initial(B)
        x = (x / (s.u @ x)[None, :]).contiguous()
        w = _NKWork(n, B, 1, x.device, s.tables.P)
        cc = torch.zeros(npr * 49 * nh ** 3, dtype=torch.float64, device="cuda")
        hg, zero = torch.zeros((B, n), dtype=torch.float64, device="cuda"), torch.zeros(B, dtype=torch.float64, device="cuda")
        st = _lib.EE0D(ns=nh, npr=npr, ccA=cc.data_ptr(), ccB=cc.data_ptr(), h=hg.data_ptr(), g=hg.data_ptr(),
                       negam=zero.data_ptr())
        bt, keep = s.batch_struct(x, n0, Tg, E, ns)
        _lib.call("bz_ee_newton_residual", s.tables.struct, bt, st, w.mu, w.F, w.fn)
        uh = s.u / torch.linalg.vector_norm(s.u)
        v = torch.from_numpy(rng.normal(size=(B, n))).cuda()
        v = (v - (v @ uh)[:, None] * uh).contiguous()
        w.active.fill_(1)
        w.active[B - 1] = 0
        w.Jz.fill_(7.0)
        _lib.call("bz_ee_newton_factor", s.tables.struct, bt, w.active, w.lprof, w.z1, w.s1)
        _lib.call("bz_ee_newton_precond_apply", s.tables.struct, bt, w.active, w.lprof, w.z1, w.s1, v, w.Jz, None)
        z = w.Jz[:B - 1]
        assert bool((w.Jz[B - 1] == 7.0).all())
        coef = torch.cat([n0[None] * ns, (n0 * Tg)[None], E[None]])
        K = sum(coef[k, :B - 1, None] * (z @ o.t()) for k, o in enumerate(list(s.C) + [s.Cg, s.A]))
        Lz = torch.linalg.solve(s.M, K.t()).t() - w.mu[:B - 1, None] * z
        Lz = Lz - (Lz @ uh)[:, None] * uh
        err = (Lz - v[:B - 1]).abs().amax(1) / v[:B - 1].abs().amax(1)
        print("pattern", pattern, "slots", s.tables.struct.nslots, "err", err.cpu().numpy(), flush=True)
        assert float(err.max()) <= 1e-7
        assert float(((z @ s.u).abs() / (s.u.abs().max() * z.abs().amax(1))).max()) <= 1e-12
