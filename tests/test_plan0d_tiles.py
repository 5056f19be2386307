"""The blocked elimination of the fused 0D solver (four pivots at a time, tiles of 16 row slots):
its slot schedule and algorithm on the host against dense LU, and the solver on tables of this
form against the one-pivot-a-step form (tables planned with the e-e pattern) on the GPU."""
import numpy as np
import pytest

from helpers import instance_params, oracle_batched, product_grid, product_xsecs
from boltzmann_amd.plan0d import permutation, plan_structure, tile_schedule


def _window(bw):
    for W in (8, 11, 12, 17, 20):
        if bw + 1 <= W:
            return W
    return -1


def _emulate(A, first, bw, W, rhs):
    """factor_tiles on the host: slots own rows by the schedule, every block of four columns
    publishes its pivot rows and updates the rows in the slots; returns U (rows) and L^-1 rhs."""
    n = A.shape[0]
    NG = (W + 2) // 4
    slot_first, sched_next, nslots = tile_schedule(first, bw, W)
    assert nslots % 64 != 0 and len(slot_first) % 64 == 0
    last = np.minimum(np.arange(n) + bw, n - 1)

    def group(row, h):                              # the four columns of group h of a row, zero outside its profile
        v = np.zeros(4)
        for q in range(4):
            c = 4 * h + q
            if row >= 0 and first[row] <= c <= last[row]:
                v[q] = A[row, c]
        return v
    ns = len(slot_first)
    read = list(slot_first)                         # row whose columns the slot reads
    comp = list(slot_first)                         # row being eliminated
    win = np.zeros((ns, NG + 1, 4))                 # panel and ring
    y = np.array([rhs[r] if r >= 0 else 0.0 for r in comp])
    for s in range(ns):
        for h in range(NG + 1):
            win[s, h] = group(read[s], h)
    U = np.zeros((n + 4, n + 4 * (NG + 2)))
    out = np.zeros(n + 4)
    for g in range((n + 3) // 4):
        P = np.eye(4, 4 * (NG + 1))
        pr = np.zeros(4)
        for s in range(ns):
            if comp[s] >= 0 and comp[s] // 4 == g:
                P[comp[s] % 4] = win[s].reshape(-1)
                pr[comp[s] % 4] = y[s]
                comp[s] = sched_next[comp[s]]
                win[s] = 0.0
                y[s] = rhs[comp[s]] if comp[s] >= 0 else 0.0
        for k in range(4):
            for i in range(k + 1, 4):
                m = P[i, k] / P[k, k]
                P[i, k:] -= m * P[k, k:]
                pr[i] -= m * pr[k]
        U[4 * g:4 * g + 4, 4 * g:4 * g + 4 * (NG + 1)] = P
        out[4 * g:4 * g + 4] = pr
        L = win[:, 0] @ np.linalg.inv(P[:, :4])
        win[:, 1:] -= (L @ P[:, 4:]).reshape(ns, NG, 4)
        y -= L @ pr
        h = g + NG + 1
        for s in range(ns):
            while read[s] >= 0 and h > read[s] // 4 + NG:
                read[s] = sched_next[read[s]]
            win[s, :-1] = win[s, 1:].copy()
            win[s, -1] = group(read[s], h)
    return U[:n, :n], out[:n]


# n = 4 k, 4 k + 1, ... and the windows 8, 11 and 17
@pytest.mark.parametrize("Nr,lmax,nproc", [(24, 1, 3), (25, 2, 3), (23, 2, 1), (24, 4, 3), (26, 1, 1), (27, 0, 3)])
def test_blocked_schedule_reproduces_lu(Nr, lmax, nproc):
    ops, g, procs = oracle_batched(Nr, lmax)
    use = range(nproc)
    mask = (np.abs(sum(ops.FOp[k] for k in use)) + np.abs(ops.FOp_g) + np.abs(ops.adv_raw) + np.abs(ops.M)) > 0
    st = plan_structure(mask, g.num_p, g.num_sh, _window)
    perm = permutation(g.num_p, g.num_sh)
    rng = np.random.default_rng(5)
    n = st["n"]
    A = np.where(mask, rng.normal(size=mask.shape), 0.0)[np.ix_(perm, perm)]
    A[np.arange(n), np.arange(n)] = 4.0 * np.sqrt(n)        # no pivoting
    b = rng.normal(size=n)
    U, y = _emulate(A, st["first_col"], st["bw"], st["W"], b)
    Ud, yd = A.copy(), b.copy()
    for j in range(n - 1):
        m = Ud[j + 1:, j] / Ud[j, j]
        Ud[j + 1:, j:] -= np.outer(m, Ud[j, j:])
        yd[j + 1:] -= m * yd[j]
    assert np.abs(U - np.triu(Ud)).max() <= 1e-13 * np.abs(Ud).max()
    assert np.abs(y - yd).max() <= 1e-13 * np.abs(yd).max()


# three, five and eight tiles, the windows 8, 11 and 17, last blocks of one to four rows; both
# forms stop at |r| <= 1e-14 |r0|, where the solutions of either agree with the fixed point to
# 1e-9 or better on these grids
@pytest.mark.gpu
@pytest.mark.parametrize("Nr,lmax,nproc,B", [(24, 1, 3, 5), (41, 2, 3, 7), (128, 1, 3, 3), (130, 2, 2, 6), (46, 4, 3, 5),
                                             (200, 2, 3, 2)])
def test_blocked_solver_equals_one_pivot_form(Nr, lmax, nproc, B):
    import torch
    from boltzmann_amd.solver0d import Batched0D
    print(f"case: blocked against one-pivot form, Nr={Nr} lmax={lmax} nproc={nproc} B={B}", flush=True)
    ops, g, procs = oracle_batched(Nr, lmax)
    vg = product_grid(g)
    xs = product_xsecs()[:nproc]
    prm = instance_params(B, seed=Nr)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()
    # E/N up to 100 Td: below the band without a root of the batched residual
    E = 10.0 ** (2.0 / 3.0 * np.log10(prm["EbyN"])) * prm["n0"] * 1e-21
    res = []
    for ee in (False, True):
        s = Batched0D(vg, xs, growth="collisions", ee_pattern=ee)
        assert (s.tables.struct.nslots % 64 == 0) == ee
        h, q, info = s.solve(d(prm["n0"]), d(prm["Tg"]), d(E), d(prm["ns_by_n0"][:nproc]), atol=0.0, rtol=1e-14,
                             max_iter=30)
        torch.cuda.synchronize()
        assert int((info["res_abs"] <= 1e-12 * info["res0"]).sum()) == B
        res.append(h.cpu().numpy())
    assert np.linalg.norm(res[0] - res[1], axis=0).max() <= 1e-9 * np.linalg.norm(res[1], axis=0).min()
