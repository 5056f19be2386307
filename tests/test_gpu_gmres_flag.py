"""The stop flag of an Arnoldi step (bz_gmres_orthogonalise): set by one workgroup of the last launch
while the others may still be reading it.

A workgroup of that launch either writes the whole of its part of V_(i+1) or nothing of it.  Its part is
the entries of every 512-entry block b with the same b mod (number of workgroups); |w| summed in any
order differs by less than n eps, the division by half an ulp."""
import ctypes

import numpy as np
import pytest
import torch

from boltzmann_amd import _lib

pytestmark = pytest.mark.gpu
THREADS = 512


def _workgroups(n):
    return 2 * max(1, min(256, (n + THREADS - 1) // THREADS))


@pytest.mark.parametrize("n", [511, 1025, 40000, 1000003])
def test_a_workgroup_writes_its_part_or_nothing(n):
    print(f"case: converging Arnoldi step, n={n}", flush=True)
    m, filler = 3, 7.0
    gen = torch.Generator(device="cuda").manual_seed(n)
    f64 = dict(dtype=torch.float64, device="cuda")
    w0 = torch.randn(n, generator=gen, **f64)
    V = torch.zeros((m + 1, n), **f64)
    V[0, 0] = 1.0
    H = torch.zeros((m + 2, m + 1), **f64)
    cs, sn, g = torch.zeros(m + 1, **f64), torch.zeros(m + 1, **f64), torch.zeros(m + 2, **f64)
    part = torch.empty((m + 1) * 256, **f64)
    tol = torch.full((1,), 1e300, **f64)                # every step converges
    flags = torch.zeros(2, dtype=torch.int32, device="cuda")
    ptr = lambda k: ctypes.c_void_p(flags.data_ptr() + 4 * k)
    part_of = (np.arange(n) // THREADS) % _workgroups(n)
    want = w0.clone()
    want[0] = 0.0                                       # the component along V_0
    want = (want / torch.linalg.vector_norm(want)).cpu().numpy()
    for rep in range(10):
        w = w0.clone()
        V[1] = filler
        g.zero_()
        g[0] = 1.0
        flags.zero_()
        _lib.call("bz_gmres_orthogonalise", V, n, m, 0, w, n, 1, part, H, m + 1, cs, sn, g, tol, ptr(0), ptr(1))
        assert flags.tolist() == [1, 1]
        row = V[1].cpu().numpy()
        kept = row == filler
        skipped = np.bincount(part_of, weights=kept, minlength=1)
        assert np.all((skipped == 0) | (skipped == np.bincount(part_of, minlength=1)))
        assert not kept[part_of == 0].any()
        assert np.abs(np.where(kept, want, row) - want).max() <= max(n, 64) * np.finfo(float).eps * np.abs(want).max()
