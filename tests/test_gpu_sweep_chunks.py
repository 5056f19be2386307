"""The chunked sweeps of bz_banded.hip at the edges of their chunks (8 and 16 positions), of a
wavefront's 64 systems and of the number of diagonals, against forward substitution on the host.

With the couplings of a row at most half its diagonal in sum, an error committed at one position is
halved by the next ones, so the result is within twice the rounding error of one position: (nd + 4)
operations on values of at most 2 max|x|, hence 4 (nd + 4) eps max|x|.
"""
import numpy as np
import pytest
import torch

from boltzmann_amd import _lib, rawkernel

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


def _dev(a):
    return torch.tensor(a, dtype=torch.float64, device="cuda")


def _substitute(diags, b, lower):
    """diags (bsz, nd, N): row i couples to i -/+ d with diags[:, d, i]."""
    bsz, nd, N = diags.shape
    x = np.zeros((bsz, N))
    for p in range(N):
        i = p if lower else N - 1 - p
        s = sum((diags[:, d, i] * x[:, i - d if lower else i + d] for d in range(1, min(nd, p + 1))), np.zeros(bsz))
        x[:, i] = (b[:, i] - s) / diags[:, 0, i]
    return x


def _close(x, y, nd):
    x = x.cpu().numpy()
    assert np.abs(x - y).max() <= 4 * (nd + 4) * EPS * np.abs(y).max()


@pytest.mark.parametrize("bsz,N,nd", [(1, 1, 1), (1, 7, 8), (63, 8, 6), (64, 9, 7), (65, 15, 2), (130, 16, 4),
                                      (64, 17, 5), (3, 33, 3), (67, 100, 8)])
@pytest.mark.parametrize("lower", [True, False])
def test_banded_and_bidiagonal(bsz, N, nd, lower):
    rng = np.random.default_rng(N + nd)
    diags = rng.uniform(-0.5, 0.5, (bsz, nd, N)) / max(nd - 1, 1)
    diags[:, 0] = rng.uniform(1.0, 2.0, (bsz, N))
    b = rng.normal(size=(bsz, N))
    ref = _substitute(diags, b, lower)
    padded = diags.copy()
    for d in range(1, min(nd, N + 1)):                  # couplings to rows outside the matrix are not used
        padded[:, d, :d] = np.nan if lower else padded[:, d, :d]
        if not lower:
            padded[:, d, max(N - d, 0):] = np.nan
    _close(rawkernel.banded_tri_solve_batched(_dev(padded), _dev(b), lower), ref, nd)
    if N > 1:
        two = np.zeros((bsz, 2, N))
        two[:, 0] = diags[:, 0]
        sub = rng.uniform(-0.5, 0.5, (bsz, N - 1))
        two[:, 1, slice(1, None) if lower else slice(0, N - 1)] = sub
        _close(rawkernel.bidiagonal_solve_batched(_dev(diags[:, 0]), _dev(sub), _dev(b), lower),
               _substitute(two, b, lower), 2)


@pytest.mark.parametrize("Nr,Nvt,Nx,nd", [(1, 1, 1, 1), (17, 3, 5, 4), (16, 8, 9, 8), (33, 2, 33, 2), (70, 6, 15, 5)])
def test_advection(Nr, Nvt, Nx, nd):
    """Both directions in one wavefront, out of place and in place."""
    rng = np.random.default_rng(Nr + nd)
    Ex, cos = rng.normal(size=Nx), rng.uniform(-1, 1, Nvt)
    vr, vx, dt = rng.uniform(0.5, 2.0, Nr), rng.uniform(0.5, 2.0, Nr), 0.3
    speed = {"vr": (-Ex[:, None] * cos[None]).reshape(-1), "vt": (Ex[:, None] / vr[None]).reshape(-1),
             "x": (vx[:, None] * cos[None]).reshape(-1)}
    for ax, fn, q, N in (("vr", rawkernel.adv_vr_BE, (Ex, cos), Nr), ("vt", rawkernel.adv_vt_BE, (Ex, vr), Nvt),
                         ("x", rawkernel.adv_x_BE, (vx, cos), Nx)):
        av = speed[ax]
        fwd = (-av >= 0) if ax == "vt" else (av >= 0)
        D = {k: rng.uniform(-0.5, 0.5, (nd, N)) / max(nd - 1, 1) for k in (True, False)}
        sign = 1.0 if ax != "vt" else -1.0
        for k in D:                                     # 1 + av dt D_0 >= 1, couplings at most half of av dt D_0
            D[k][0] = (sign if k else -sign) * rng.uniform(1.0, 2.0, N)
        b = rng.normal(size=(av.size, N))
        ref = np.zeros_like(b)
        for k in D:
            rows = fwd == k
            diags = np.zeros((rows.sum(), nd, N))
            for d in range(nd):
                for i in range(N):
                    j = i - d if k else i + d
                    if 0 <= j < N:
                        diags[:, d, i] = av[rows] * dt * D[k][d, j]
            diags[:, 0] = 1.0 + av[rows, None] * dt * D[k][0]
            ref[rows] = _substitute(diags, b[rows], k)
        out = torch.full(b.shape, float("nan"), dtype=torch.float64, device="cuda")
        args = (_dev(D[True]), _dev(D[False]), _dev(q[0]), _dev(q[1]), dt)
        fn(*args, _dev(b), out, nd, Nr, Nvt, Nx)
        _close(out, ref, nd)
        same = _dev(b)
        fn(*args, same, same, nd, Nr, Nvt, Nx)
        assert torch.equal(same, out)


def test_long_x_lines():
    """Lines past the scan's 1024 positions: both directions, the inflow value taken as zero."""
    Nr, Nvt, Nx = 2, 3, 1030
    rng = np.random.default_rng(5)
    diag, sub = rng.uniform(1.0, 2.0, (Nr * Nvt, Nx)), rng.uniform(-0.5, 0.5, (Nr * Nvt, Nx - 1))
    b, low = rng.normal(size=(Nr * Nvt, Nx)), np.array([1, 0, 1])
    ref = np.zeros_like(b)
    for s in range(Nr * Nvt):
        two, r = np.zeros((1, 2, Nx)), b[s:s + 1].copy()
        f = bool(low[s % Nvt])
        two[:, 0] = diag[s]
        two[:, 1, slice(1, None) if f else slice(0, Nx - 1)] = sub[s]
        r[0, 0 if f else -1] = 0.0
        ref[s] = _substitute(two, r, f)[0]
    out = torch.empty(b.shape, dtype=torch.float64, device="cuda")
    _lib.call("bz_xstep_bidiag_solve", _dev(diag), _dev(sub), torch.tensor(low, dtype=torch.int32, device="cuda"),
              _dev(b), out, Nr, Nvt, Nx)
    _close(out, ref, 2)


def test_very_long_lines():
    """Lines too long for the 32-bit offsets of a workgroup's results."""
    from scipy.linalg import solve_banded
    N = (1 << 20) + 3
    rng = np.random.default_rng(9)
    diag, sub, b = rng.uniform(1.0, 2.0, (2, N)), rng.uniform(-0.5, 0.5, (2, N - 1)), rng.normal(size=(2, N))
    x = rawkernel.bidiagonal_solve_batched(_dev(diag), _dev(sub), _dev(b), True)
    ref = np.stack([solve_banded((1, 0), np.stack([diag[s], np.append(sub[s], 0.0)]), b[s]) for s in range(2)])
    _close(x, ref, 2)
