"""The quotient of the advection sweeps is that of a division: rounded once, with the division's
infinities and NaN.

One diagonal, so that a position is b / (1 + av dt D_0) with nothing before it; speeds, steps and
coefficients of few bits, so that the denominator is exact in FP64 and the quotient is NumPy's."""
import numpy as np
import pytest
import torch

from boltzmann_amd import rawkernel

pytestmark = pytest.mark.gpu


def _dev(a):
    return torch.tensor(a, dtype=torch.float64, device="cuda")


@pytest.mark.parametrize("special", [False, True])
def test_quotient_of_a_position(special):
    rng = np.random.default_rng(12)
    Nr, Nvt, Nx, dt = 33, 6, 18, 0.25
    few = lambda lo, hi, n: rng.integers(lo, hi, n) / 64.0
    Ex = few(-200, 200, Nx)
    cos = np.array([-0.75, -0.5, -0.25, 0.25, 0.5, 0.75])
    vr, vx = 2.0 ** rng.integers(-2, 3, Nr), few(1, 200, Nr)
    if special:
        Ex[1], cos[1] = 8.0, 0.5                        # radial lines with av dt = -1
    speed = {"vr": (-Ex[:, None] * cos[None]).reshape(-1), "vt": (Ex[:, None] / vr[None]).reshape(-1),
             "x": (vx[:, None] * cos[None]).reshape(-1)}
    for ax, fn, q, N in (("vr", rawkernel.adv_vr_BE, (Ex, cos), Nr), ("vt", rawkernel.adv_vt_BE, (Ex, vr), Nvt),
                         ("x", rawkernel.adv_x_BE, (vx, cos), Nx)):
        av = speed[ax]
        fwd = (-av >= 0) if ax == "vt" else (av >= 0)
        DL, DR = few(1, 300, (1, N)), few(1, 300, (1, N))
        b = rng.normal(size=(av.size, N))
        if special:
            flat = b.reshape(-1)
            flat[::7], flat[1::7], flat[2::7], flat[3::7] = np.inf, np.nan, 1.7e308, -1.7e308
            DL[0, 0] = DR[0, -1] = 0.0
            if ax == "vr":                              # a zero and a small denominator
                DL[0, 1] = DR[0, 1] = 1.0
                DL[0, 2] = DR[0, 2] = 1.0 + 2.0 ** -40
        D = np.where(fwd[:, None], DL, DR)
        with np.errstate(all="ignore"):
            den = 1.0 + (av[:, None] * dt) * D
            want = b / den
        out = torch.empty(b.shape, dtype=torch.float64, device="cuda")
        fn(_dev(DL), _dev(DR), _dev(q[0]), _dev(q[1]), dt, _dev(b), out, 1, Nr, Nvt, Nx)
        np.testing.assert_array_equal(out.cpu().numpy(), want, err_msg=ax)
