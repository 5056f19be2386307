"""The path that the ion-fluid launch takes at sizes of the 4 x 4 tile layout (up to 88 points) and the
next one, by the column ratio of the Jacobian J = I + h Dp (mu diag(E) - Di Dp_mod): Jacobi iterations
up to 0.5, the tile inverse between 0.5 and 1, the pivoted inverse where a column is not
dominant; each against the oracle's step with the tolerances of test_fluid_launch_against_oracle."""
import numpy as np
import pytest
import torch

from oracle import glow_coupled as gc
from test_gpu_glow_coupled import _glow, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Np", [20, 50, 75, 88, 89])
def test_paths(Np):
    from boltzmann_amd.glowdischarge_boltzmann_1d import GLOW_FIELD_AFTER, GLOW_STEP
    glow = _glow(8, 1, Np, 4, 1e-3)
    glow._setup_fluid()
    p, xp = glow.param, glow.xp
    s = 0.5 * (xp + 1)
    mu, Di = np.full(Np, p.mu_i), np.full(Np, p.Di)
    ne = 1e6 * (1e7 + 1e9 * s ** 2 * (1 - s) ** 2) / p.np0 * (1 + 0.02 * np.cos(5 * xp))
    ni = ne * (1 + 0.03 * np.sin(3 * np.pi * xp))
    ki = 2e-3 * (1.5 + 0.5 * np.cos(2 * xp))
    u = np.stack([ne, ni, np.full(Np, 3.0)], axis=1)
    glow._ki.copy_(torch.from_numpy(ki))
    t0 = 0.137

    def launch(h):
        ud = torch.from_numpy(u.copy()).cuda()
        glow._fluid_launch(ud, GLOW_STEP | GLOW_FIELD_AFTER, h=h, t_before=t0, t_after=t0 + h)
        torch.cuda.synchronize()
        return ud, glow._status.tolist(), glow._Ef.cpu().numpy()

    Dp_mod = np.array(glow.Dp)
    Dp_mod[0] = Dp_mod[-1] = 0.0
    E = launch(1e-9)[2]
    A = np.array(glow.Dp) @ (np.diag(p.mu_i * E) - p.Di * Dp_mod)

    def ratio(h):
        J = np.eye(Np) + h * A
        d = np.abs(np.diag(J))
        return float(((np.abs(J).sum(axis=0) - d) / d).max())

    ran = []
    for want, path in ((0.25, 4), (0.75, 0), (3.0, 2)):
        lo, hi = 1e-9, 1.0
        for _ in range(60):                             # the ratio starts at zero
            mid = np.sqrt(lo * hi)
            lo, hi = (mid, hi) if ratio(mid) < want else (lo, mid)
        h = lo
        if not 0.5 * want < ratio(h) < 1.3 * want:
            continue
        ud, st, E1 = launch(h)
        print(f"case: Np={Np} h={h:.3e} column ratio {ratio(h):.3f} status {st}", flush=True)
        assert st[0] == 1 and (st[3] & 1) == 0, st
        assert (st[3] & 6) == path
        ran.append(path)
        np.testing.assert_array_equal(E1, E)
        r = -p.alpha * (ni - ne)
        r[0], r[-1] = np.sin(2 * np.pi * t0), 0.0
        kappa = float((np.abs(glow.Dp) @ (np.abs(glow.LpD_inv) @ np.abs(r))).max() / np.abs(E).max())
        tol_E = 20 * 2.2e-16 * kappa
        Eo = glow.Dp @ (-gc.solve_poisson(glow.LpD_inv, p.alpha, ne, ni, t0))
        assert _rel(E, Eo) < tol_E
        u1, info = gc.step_fluid_be(glow.Dp, mu, Di, p.n0, ki, Eo, u, h, glow.args.atol, glow.args.rtol,
                                    glow.args.max_iter)
        dn = _rel(ud[:, 1] - torch.from_numpy(ni).cuda(), u1[:, 1] - ni)
        assert _rel(ud[:, 1], u1[:, 1]) < max(1e-13, tol_E)
        assert dn < max(1e-11, 10 * tol_E)
    assert 4 in ran and 0 in ran, ran
