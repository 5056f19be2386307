"""Restarted, right-preconditioned GMRES on the device.

Mirrors utils.gmres_pcr (BESolver/python/utils.py:1172-1268): same arguments, same
right preconditioning (A M^-1 y = b, x = M^-1 y), the least-squares problem of the
Hessenberg matrix solved after every Arnoldi step, a true-residual check b - A M^-1 x_n
after every step, tol = max(atol, rtol |b|), maxiter tested between restart cycles only (a
cycle always runs to its end), return value (solution, info) with info 0 on convergence and
the iteration count otherwise.

Design: the Krylov basis lives in HBM as rows of one (restart+1, n) array; every
Arnoldi step is two block dot products and two block updates (classical Gram-Schmidt
applied twice - the reference uses modified Gram-Schmidt; both give an orthonormal
basis to FP64 rounding), one norm and one scaling, all in HIP kernels
(bz_krylov.hip).  The Hessenberg least-squares problem is solved on the device by
Givens rotations.  The host reads one scalar per step (the true residual norm), as
the reference does.
"""
import ctypes
import gc
import inspect

import torch

from . import _lib


def _at(t, offset=0):
    """Device address of element `offset` of a contiguous tensor (for strided views the
    kernels take an explicit stride)."""
    assert t.is_cuda and t.is_contiguous()
    return ctypes.c_void_p(t.data_ptr() + 8 * offset)


class _Work:
    def __init__(self, n, restart, dev):
        self.n = n
        self.nblk = max(1, min(1024, (n + 4095) // 4096))
        self.V = torch.empty((restart + 1, n), dtype=torch.float64, device=dev)
        self.H = torch.zeros((restart + 2, restart + 1), dtype=torch.float64, device=dev)
        self.ldh = restart + 1
        self.partial = torch.empty(((restart + 1) * self.nblk,), dtype=torch.float64, device=dev)
        self.h = torch.zeros(restart + 2, dtype=torch.float64, device=dev)
        self.scal = torch.zeros(4, dtype=torch.float64, device=dev)
        self.lsq_R = torch.empty(((restart + 2) * (restart + 1),), dtype=torch.float64, device=dev)
        self.lsq_y = torch.empty((2 * restart + 2,), dtype=torch.float64, device=dev)
        self.u = torch.empty(n, dtype=torch.float64, device=dev)

    def dot(self, V, nv, u, out, ostride=1, accumulate=0, take_sqrt=0, out2=None):
        _lib.call("bz_multi_dot", _at(V), self.n, nv, _at(u), self.n, self.partial, self.nblk, out, ostride, accumulate,
                  take_sqrt, out2)

    def norm(self, x):
        """|x| into scal[0] (device); returns that 1-element view."""
        self.dot(x, 1, x, _at(self.scal), take_sqrt=1)
        return self.scal[0:1]


def gmres_pcr(A, b, x0=None, atol=1e-20, rtol=1e-10, maxiter=None, restart=None, M=None, callback=None):
    """A, M: objects with .matvec(x) on flat device vectors (or callables); b a flat
    float64 device vector.  Returns (x, info)."""
    n = b.numel()
    if n == 0:
        return torch.empty_like(b), 0
    matvec = A.matvec if hasattr(A, "matvec") else A
    psolve = (M.matvec if hasattr(M, "matvec") else M) if M is not None else (lambda v: v)
    if maxiter is None:
        maxiter = n * 10
    if restart is None:
        restart = maxiter
    restart = int(restart)
    w = _Work(n, restart, b.device)
    b = b.contiguous()
    b_norm = float(w.norm(b).item())
    if b_norm == 0:
        return b, 0
    tol = max(atol, rtol * b_norm)
    x = torch.zeros_like(b) if x0 is None else x0.reshape(-1).contiguous().clone()
    V, H, ldh = w.V, w.H, w.ldh
    beta = torch.zeros(1, dtype=torch.float64, device=b.device)
    it = 0
    xn = x
    while it < maxiter:
        H.zero_()
        mx = psolve(x)
        r = (b - matvec(mx)).contiguous()
        beta.copy_(w.norm(r))
        if float(beta.item()) < tol:
            return mx, 0
        _lib.call("bz_scale_inv", r, beta, _at(V, 0), n)
        for i in range(restart):
            w.u.copy_(matvec(psolve(V[i])))
            # H[0:i+1, i] = V^T u, applied twice (classical Gram-Schmidt, re-orthogonalised)
            for rep in range(2):
                w.dot(V, i + 1, w.u, _at(H, i), ostride=ldh, accumulate=rep, out2=w.h)
                _lib.call("bz_vt_axpy", _at(V), n, i + 1, w.h, 1, -1.0, w.u, w.u, n)
            w.dot(w.u, 1, w.u, _at(H, (i + 1) * ldh + i), take_sqrt=1)
            _lib.call("bz_scale_inv", w.u, _at(H, (i + 1) * ldh + i), _at(V, (i + 1) * n), n)
            _lib.call("bz_hess_lstsq", H, ldh, i + 1, beta, w.lsq_R, w.lsq_y)
            xn = torch.empty_like(x)
            _lib.call("bz_vt_axpy", _at(V), n, i + 1, w.lsq_y, 1, 1.0, x, xn, n)
            rn = (b - matvec(psolve(xn))).contiguous()
            rn_norm = float(w.norm(rn).item())
            if callback is not None:
                callback(rn_norm / b_norm)
            if rn_norm < tol:
                return psolve(xn), 0
            it += 1
        x = xn
    return psolve(xn), it + 1


def _ptr(t, offset=0):
    """Device address of element `offset` of a contiguous tensor of any element type."""
    assert t.is_cuda and t.is_contiguous()
    return ctypes.c_void_p(t.data_ptr() + t.element_size() * offset)


class capture_guard:
    """Collects dead Python reference cycles before a stream capture and keeps the cyclic
    garbage collector off during it.  A dead cycle can hold captured graphs or device memory
    (a solver and its GMRES object referring to each other); if the collector frees them in
    the middle of another capture, the graph's teardown and the freeing of its memory pool
    are device calls that a capturing stream does not allow, and the process aborts.  This
    torch release no longer collects at the start of a capture by default."""

    def __enter__(self):
        gc.collect()
        self._was = gc.isenabled()
        gc.disable()
        return self

    def __exit__(self, *exc):
        if self._was:
            gc.enable()
        return False


class ArnoldiCycle:
    """The device state of a restarted GMRES cycle and its vector operations (bz_krylov.hip):
    basis, Hessenberg column rotation, residual estimate, stop flag.  A subclass supplies
    `product(src, out, done)`: t = P src and out = A t (device addresses; nothing when the device
    flag `done` is set).  After the first cycle everything between two read-backs is one HIP graph:
    the residual of a start vector, the beginning of a cycle with its first `chunk` steps, each
    further chunk, and the end of a cycle (solution and true residual).  The host reads the stop
    flag after a chunk and the residual after a cycle.  Steps past convergence are no-ops."""

    def __init__(self, n, restart, dev, chunk, gs_passes, use_graph=True):
        f64, i32 = torch.float64, torch.int32
        self.n, self.m, self.chunk = int(n), int(restart), int(chunk)
        self.gs_passes = int(gs_passes)                             # classical Gram-Schmidt passes
        self.use_graph = use_graph
        m = self.m
        self.V = torch.zeros((m + 1, self.n), dtype=f64, device=dev)
        self.H = torch.zeros((m + 2, m + 1), dtype=f64, device=dev)
        self.ldh = m + 1
        self.partial = torch.empty(((m + 1) * 256,), dtype=f64, device=dev)
        self.cs = torch.zeros(m + 1, dtype=f64, device=dev)
        self.sn = torch.zeros(m + 1, dtype=f64, device=dev)
        self.g = torch.zeros(m + 2, dtype=f64, device=dev)
        self.tol = torch.zeros(1, dtype=f64, device=dev)
        self.stat = torch.zeros(4, dtype=f64, device=dev)           # |r|, |b|, tolerance, steps
        self.flags = torch.zeros(2, dtype=i32, device=dev)          # done, steps of the cycle
        self.w, self.t, self.x, self.b, self.r = (torch.empty(self.n, dtype=f64, device=dev) for _ in range(5))
        self.graphs = None

    def _step(self, i):
        done, kdone = _ptr(self.flags, 0), _ptr(self.flags, 1)
        self.product(_at(self.V, i * self.n), _at(self.w), done)
        _lib.call("bz_gmres_orthogonalise", self.V, self.n, self.m, i, self.w, self.n, self.gs_passes, self.partial,
                  self.H, self.ldh, self.cs, self.sn, self.g, self.tol, done, kdone)

    def _steps(self, i0):
        for i in range(i0, min(self.m, i0 + self.chunk)):
            self._step(i)

    def _capture(self, parts):
        """The replays of one graph for every sequence of launches in `parts`."""
        run = {}
        with capture_guard():
            for name, launch in parts.items():
                gr = torch.cuda.CUDAGraph()
                with torch.cuda.graph(gr):
                    launch()
                run[name] = gr.replay
        return run

    def _norm(self, of, b, ax, r, atol=0.0, rtol=0.0):
        _lib.call("bz_gmres_norm", b, ax, r, self.n, self.partial, of, float(atol), float(rtol), _ptr(self.flags, 1),
                  self.stat)

    def _residual(self):
        """r = b - A P x with its norm; leaves P x in t."""
        self.product(_at(self.x), _at(self.r), None)
        self._norm(0, self.b, self.r, self.r)

    def _solution(self):
        """x += V y over the steps of the cycle."""
        if self.m > 8000:                                           # more rows of y than fit the kernel's LDS
            y = torch.zeros(self.m, dtype=torch.float64, device=self.x.device)
            _lib.call("bz_gmres_back_solve", self.H, self.ldh, self.g, _ptr(self.flags, 1), y, self.m)
            _lib.call("bz_gmres_add", self.V, self.n, y, _ptr(self.flags, 1), self.x, self.n)
            return
        _lib.call("bz_gmres_solution", self.V, self.n, self.m, self.H, self.ldh, self.g, _ptr(self.flags, 1), self.x,
                  self.n)

    def cycles(self, atol, rtol, max_cycles, zero_start, callback=None):
        """Cycles from x (zero_start: x = 0) for the right-hand side b, until the true residual
        is below tol = max(atol, rtol |b|).  Returns (converged, total steps); P x is in t."""
        def begin():
            # r and its norm are those of the current x: from the start, or from the end of the
            # previous cycle.  When |r| is below the tolerance at the start the cycle is empty.
            _lib.call("bz_gmres_begin", self.r, self.stat, self.V, self.n, self.m, self.g, self.tol,
                      _ptr(self.flags, 0), _ptr(self.flags, 1))
            self._steps(0)

        def end():
            self._solution()
            self._residual()

        parts = {"residual": self._residual, "end": end, 0: begin}
        parts.update({i0: lambda i0=i0: self._steps(i0) for i0 in range(self.chunk, self.m, self.chunk)})
        run = self.graphs or parts
        if zero_start:
            self.t.zero_()
            self._norm(2, self.b, None, self.r, atol, rtol)        # r = b
        else:
            self._norm(1, self.b, None, None, atol, rtol)
            run["residual"]()
        iters = 0
        for _ in range(max_cycles):
            for i0 in range(0, self.m, self.chunk):
                run[i0]()
                if int(self.flags[0].item()):
                    break
            run["end"]()
            if self.graphs is None and self.use_graph:
                # the eager cycle has loaded and run every kernel once
                self.graphs = run = self._capture(parts)
            # one read-back per cycle: the true residual, |b|, the tolerance and the step count
            rn, bn, tol, k = self.stat.tolist()
            iters += int(k)
            if callback is not None and k > 0:                     # not for a start that is already converged
                callback(rn / bn if bn > 0 else 0.0)
            if rn < tol:
                return True, iters
        return False, iters


def _with_flag(launch):
    """A launcher (src, dst, done) of one that takes (src, dst) or already the flag.  Without the
    flag it overwrites dst in steps past convergence too, which nothing reads."""
    if launch is None:
        return None
    try:
        inspect.signature(launch).bind(None, None, None)
        return launch
    except (TypeError, ValueError):
        return lambda src, dst, done: launch(src, dst)


class DeviceGMRES(ArnoldiCycle):
    """Restarted, right-preconditioned GMRES with the whole Arnoldi step on the device, for an
    operator and a preconditioner given as launchers `matvec(src, dst)` and `precond(src, dst)`
    (device addresses of flat float64 vectors of length n; each writes dst only).  A launcher that
    takes a third argument is given the device flag `done` and may write nothing when it is set
    (it is None outside a cycle): steps past convergence then cost their launches only.

    The method of utils.gmres_pcr (utils.py:1172-1268: right preconditioning, restart,
    tol = max(atol, rtol |b|)) with the host out of the inner loop: the stop test of a step
    is the least-squares residual |g_(i+1)| of the Givens-rotated Hessenberg system (the
    true residual in exact arithmetic), and the true residual is evaluated once per cycle, at its
    end, before the solution is accepted.  Per step: preconditioner, operator and
    bz_gmres_orthogonalise (classical Gram-Schmidt, two passes by default, one with gs_passes=1).
    The launchers' scalar arguments and buffers are captured with the graphs, so they must stay
    the same between solves (inputs are copied into fixed buffers)."""

    def __init__(self, n, restart, dev, matvec, precond, chunk=4, use_graph=True, gs_passes=2):
        super().__init__(n, restart, dev, chunk, gs_passes, use_graph)
        self.matvec, self.precond = _with_flag(matvec), _with_flag(precond)

    def product(self, src, out, done):
        self.precond(src, _at(self.t), done)
        self.matvec(_at(self.t), out, done)

    def solve(self, b, atol, rtol, max_cycles, x0=None, callback=None):
        """Returns (P x, total steps); raises RuntimeError after max_cycles cycles."""
        self.b.copy_(b.reshape(-1))
        if x0 is None:
            self.x.zero_()
        else:
            self.x.copy_(x0.reshape(-1))
        converged, iters = self.cycles(atol, rtol, max_cycles, x0 is None, callback)
        if not converged:
            raise RuntimeError(f"GMRES did not converge in {max_cycles} cycles of {self.m}")
        return self.t.clone(), iters
