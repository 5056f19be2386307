"""Patterns whose blocked schedule needs every slot of the largest solver instance."""
import types

import numpy as np
import pytest

from boltzmann_amd import plan0d
from boltzmann_amd.plan0d import plan_structure, tile_schedule

N, FULL = 260, 192


def _pattern(full=FULL):
    """(permuted order) the first `full` rows start at column 0, the rest keep three columns."""
    first = np.where(np.arange(N) < full, 0, np.arange(N) - 3)
    return np.array([[first[i] <= j <= i + 3 for j in range(N)] for i in range(N)])


def _mask(full=FULL):
    perm = plan0d.permutation(N, 1)
    m = np.zeros((N, N), bool)
    m[np.ix_(perm, perm)] = _pattern(full)
    return m


@pytest.mark.parametrize("full", [FULL - 1, FULL, 64, 65])
def test_schedule_fits_the_solver(full):
    """One-pivot tables have nslots a multiple of 64, blocked ones not, and neither passes the
    slots of the largest instance when its rows fit them."""
    st = plan_structure(_mask(full), N, 1, lambda bw: 8)
    first, nxt, nslots = plan0d.solver_schedule(st, False)
    assert nslots <= FULL and len(first) % 64 == 0 and len(first) >= nslots
    blocked = tile_schedule(st["first_col"], st["bw"], st["W"])
    assert (nslots % 64 == 0) == (full == FULL)
    if full == FULL:
        assert blocked[2] == FULL + 1 and nslots == st["nslots"]
    else:
        assert nslots == blocked[2]


@pytest.mark.gpu
def test_both_planners_and_the_solver_take_it():
    import torch
    from boltzmann_amd import _lib
    from boltzmann_amd.plan0d import CPlannedGrid, SolverTables
    print("case: 192 slots, both planners, two Newton steps", flush=True)
    rng = np.random.default_rng(0)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()
    band = np.abs(np.arange(N)[:, None] - np.arange(N)[None]) <= 3
    M = np.eye(N) + 0.05 * band
    full = _mask()
    C0 = np.where(full, -0.01 * rng.uniform(0.5, 1.0, (N, N)), 0.0) - 2.0 * np.eye(N)
    ops = [d(C0), d(np.where(band, 0.01, 0.0)), d(np.where(band, 0.02, 0.0)), d(M)]
    u, mass = d(rng.uniform(0.5, 1.0, N)), d(M)
    grid = types.SimpleNamespace(dev=torch.device("cuda", 0), npr=N, num_sh=1, n=N)
    tables = SolverTables(grid, ops, [True, False, False], u, mass)
    planned = CPlannedGrid(grid, ops, [ops[0], None, None], u, mass)
    B, outs = 3, []
    one = torch.ones(B, dtype=torch.float64, device="cuda")
    for t in (tables, planned):
        assert t.struct.nslots == FULL
        f = lambda *s: torch.zeros(s, dtype=torch.float64, device="cuda")
        x = d(rng.uniform(0.9, 1.1, (N, B))) if not outs else outs[0][1].clone()
        x0 = x.clone()
        sc = (f(B, tables.P), f(B, N * tables.WP), f(B, plan0d.VEC_ROWS, N), f(B), f(B))
        it, st = (torch.zeros(B, dtype=torch.int32, device="cuda") for _ in range(2))
        bt = _lib.Batch0D(B=B, n0=one.data_ptr(), Tg=one.data_ptr(), E=one.data_ptr(), ns_by_n0=one.data_ptr(),
                          x=x.data_ptr(), kprof=sc[0].data_ptr(), urows=sc[1].data_ptr(), vec=sc[2].data_ptr(),
                          iters=it.data_ptr(), status=st.data_ptr(), res_abs=sc[3].data_ptr(), res0=sc[4].data_ptr(),
                          atol=0.0, rtol=1e-12, alpha_min=1e-16, alpha_rho=0.5, ls_c=1e-4, max_iter=2, mode=1,
                          tg_scale=1.0, tol_abs=None)
        _lib.call("bz_steady_solve_0d", t.struct, bt)
        torch.cuda.synchronize()
        outs.append((x, x0))
        assert bool(torch.isfinite(x).all())
    assert torch.equal(outs[0][0], outs[1][0])
