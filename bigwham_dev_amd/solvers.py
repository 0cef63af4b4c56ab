"""Krylov solvers around the MI355X H-matvec (the caller side of the path).

The reference ships no solver: users call scipy.sparse.linalg.gmres on the
BEMatrix LinearOperator with the Jacobi preconditioner 1/diag(H)
(interfaces/python/bigwham4py/bigwham4py.py:362-380), one host<->device round
trip per iteration on the CUDA path.  Here GMRES runs on the device with
torch FP64 vectors:

  gmres()        restarted right-preconditioned GMRES, FP64 Arnoldi with
                 classical Gram-Schmidt and one re-orthogonalisation pass,
                 Givens rotations on the host.
  solve_mixed()  mixed precision: iterative refinement whose residual
                 r = b - H x is evaluated with the FP64 matvec and whose
                 correction solves H d = r with gmres() driven by the
                 FP32-factor matvec (FP64 Arnoldi and vectors),
                 restarting from the Arnoldi residual; stops on the FP64
                 residual.
"""
from __future__ import annotations

import ctypes as C
import math
import time
from dataclasses import dataclass, field

import torch
from torch.autograd import forward_ad

from . import _native as N


@dataclass
class SolveInfo:
    converged: bool
    iterations: int           # total inner matvecs
    matvecs_fp64: int
    matvecs_fp32: int
    rel_residual: float       # ||b - H64 x|| / ||b|| at exit
    seconds: float
    history: list = field(default_factory=list)


def gmres(matvec, b: torch.Tensor, precond=None, x0: torch.Tensor | None = None,
          tol: float = 1e-8, restart: int = 30, maxiter: int = 1000,
          callback=None, implicit_restart: bool = False):
    """Solve A x = b; matvec(v) -> A v on device (float64).  precond(v) -> M^{-1} v
    (right preconditioning).  Returns (x, iterations, rel_residual_estimate).

    Each iteration synchronises with the host once (the Hessenberg column and
    the new basis norm come back together); the basis vector itself is
    normalised on the device, and on the GPU the next iteration is already
    queued when the host waits.  A restart recomputes the residual b - A x with
    one matvec, or, with ``implicit_restart``, forms it from the Arnoldi
    relation r = V_{m+1} (beta e_1 - Hbar y) without a matvec (used by the
    inner solves of the mixed-precision refinement, whose outer loop
    recomputes the true FP64 residual anyway)."""
    dev, dt = b.device, b.dtype
    n = b.numel()
    bnorm = torch.linalg.vector_norm(b).item()
    if bnorm == 0.0:
        return torch.zeros_like(b), 0, 0.0
    x = torch.zeros_like(b) if x0 is None else x0.clone()
    M = precond if precond is not None else (lambda v: v)
    V = torch.empty((restart + 1, n), dtype=dt, device=dev)
    # On the GPU the Hessenberg columns come back through pinned memory behind
    # events, and the next iteration (matvec and orthogonalisation) is queued
    # before the host waits for one, so the device is not left idle while the
    # host applies the rotations.
    steps = _DeviceSteps(V) if b.is_cuda else _HostSteps(V)
    try:
        return _cycles(matvec, M, b, x0, x, V, steps, bnorm, tol, restart, maxiter, callback,
                       implicit_restart)
    finally:
        steps.close()


class _HostSteps:
    """Orthogonalisation steps with torch: classical Gram-Schmidt with one
    re-orthogonalisation pass, as matrix-vector products."""

    ahead = False  # steps are done when queued: nothing to look ahead for

    def __init__(self, V):
        self.V = V

    def _torch_step(self, k, w):
        Vk = self.V[: k + 1]
        h = Vk @ w
        w = torch.addmv(w, Vk.t(), h, alpha=-1.0)
        h2 = Vk @ w
        w = torch.addmv(w, Vk.t(), h2, alpha=-1.0)
        hn = torch.linalg.vector_norm(w)
        torch.div(w, hn, out=self.V[k + 1])
        return torch.cat([h + h2, hn.reshape(1)])

    def queue(self, k, w):
        """Orthogonalise w against V[0..k] into V[k + 1]."""
        self.col = self._torch_step(k, w)

    def column(self, k):
        """Hessenberg column k: k + 1 coefficients and the norm of the rest."""
        return self.col.tolist()

    def close(self):
        pass


class _DeviceSteps(_HostSteps):
    """The same on the GPU, queued: four kernels per step
    (bw_hip_orthogonalize) that write the column to pinned memory."""

    ahead = True

    def __init__(self, V):
        super().__init__(V)
        restart, n = V.shape[0] - 1, V.shape[1]
        self.n, self.index = n, V.get_device()
        # two rows, as two steps are in flight at most; a step that a cycle left
        # behind is done before the next cycle's steps, on the same stream
        self.cols = torch.empty((2, restart + 2), dtype=V.dtype, pin_memory=True)
        self.events = [torch.cuda.Event() for _ in range(2)]
        self.queued = -1
        self.native = None
        if V.dtype == torch.float64:
            need = C.c_int64()
            if N.hip().bw_hip_orthogonalize_work(n, restart, C.byref(need)) == N.BW_OK:
                self.native = N.hip()
                self.work = torch.empty(need.value, dtype=V.dtype, device=V.device)

    def _plain(self, w):
        """Whether w is one contiguous vector of V's kind that can be read through its
        pointer: its memory holds its values (no pending negation, no subclass
        with a meaning of its own) and nothing differentiates through the step.
        Everything else is left to torch, which computes it or refuses it."""
        V = self.V
        return (type(w) is torch.Tensor and w.dtype is V.dtype and w.get_device() == self.index
                and w.dim() == 1 and w.numel() == self.n and w.is_contiguous()
                and not w.is_neg()
                and not ((w.requires_grad or V.requires_grad) and torch.is_grad_enabled())
                and (forward_ad._current_level < 0  # no dual numbers about
                     or (forward_ad.unpack_dual(w).tangent is None
                         and forward_ad.unpack_dual(V).tangent is None)))

    def queue(self, k, w):
        V = self.V
        if self.native and self._plain(w):
            rc = self.native.bw_hip_orthogonalize(
                V.device.index, V.shape[1], k + 1, V.data_ptr(), V.stride(0), w.data_ptr(),
                V[k + 1].data_ptr(), self.cols[k & 1].data_ptr(), self.work.data_ptr(),
                self.work.numel(), torch.cuda.current_stream(V.device).cuda_stream)
            if rc != N.BW_OK:
                raise N.BigWhamError(rc, "orthogonalize")
        else:
            self.cols[k & 1, : k + 2].copy_(self._torch_step(k, w), non_blocking=True)
        self.events[k & 1].record(torch.cuda.current_stream(V.device))
        self.queued = k

    def column(self, k):
        self.events[k & 1].synchronize()
        return self.cols[k & 1, : k + 2].tolist()

    def close(self):
        # a queued step still writes the pinned columns
        if self.queued >= 0:
            self.events[self.queued & 1].synchronize()


def _cycles(matvec, M, b, x0, x, V, steps, bnorm, tol, restart, maxiter, callback,
            implicit_restart):
    """The restart cycles of gmres()."""
    dev, dt = b.device, b.dtype
    its = 0
    rel = 1.0
    r = b.clone() if x0 is None else b - matvec(x)
    while its < maxiter:
        beta = torch.linalg.vector_norm(r).item()
        rel = beta / bnorm
        if rel <= tol:
            break
        V[0] = r / beta
        Hs = [[0.0] * restart for _ in range(restart + 1)]
        Hraw = [[0.0] * restart for _ in range(restart + 1)]
        cs, sn = [0.0] * restart, [0.0] * restart
        g = [0.0] * (restart + 1)
        g[0] = beta
        k_done = 0
        breakdown = False
        queued = -1
        for k in range(restart):
            if queued < k:
                steps.queue(k, matvec(M(V[k])))
                queued = k
            its += 1
            # look ahead unless the cycle ends here or the last estimate is
            # already near the tolerance (a look-ahead past convergence is
            # one wasted matvec)
            if steps.ahead and k + 1 < restart and its < maxiter and rel > 1.5 * tol:
                steps.queue(k + 1, matvec(M(V[k + 1])))
                queued = k + 1
            col = steps.column(k)
            hn = col[k + 1]
            for i in range(k + 2):
                Hs[i][k] = Hraw[i][k] = col[i]
            for i in range(k):
                t = cs[i] * Hs[i][k] + sn[i] * Hs[i + 1][k]
                Hs[i + 1][k] = -sn[i] * Hs[i][k] + cs[i] * Hs[i + 1][k]
                Hs[i][k] = t
            den = math.hypot(Hs[k][k], Hs[k + 1][k])
            cs[k] = Hs[k][k] / den if den else 1.0
            sn[k] = Hs[k + 1][k] / den if den else 0.0
            Hs[k][k] = cs[k] * Hs[k][k] + sn[k] * Hs[k + 1][k]
            Hs[k + 1][k] = 0.0
            g[k + 1] = -sn[k] * g[k]
            g[k] = cs[k] * g[k]
            k_done = k + 1
            rel = abs(g[k + 1]) / bnorm
            if callback is not None:
                callback(its, rel)
            breakdown = hn == 0.0
            if rel <= tol or its >= maxiter or breakdown:
                break
        # back substitution
        y = [0.0] * k_done
        for i in range(k_done - 1, -1, -1):
            s_ = g[i] - sum(Hs[i][j] * y[j] for j in range(i + 1, k_done))
            y[i] = s_ / Hs[i][i]
        yt = torch.tensor(y, dtype=dt, device=dev)
        x = x + M(V[:k_done].T @ yt)
        if rel <= tol or its >= maxiter:
            break
        if implicit_restart:
            m1 = k_done if breakdown else k_done + 1
            c = [(beta if i == 0 else 0.0) - sum(Hraw[i][j] * y[j] for j in range(k_done))
                 for i in range(m1)]
            r = V[:m1].T @ torch.tensor(c, dtype=dt, device=dev)
        else:
            r = b - matvec(x)
    return x, its, rel


def _sync(t: torch.Tensor) -> None:
    if t.is_cuda:
        torch.cuda.synchronize(t.device)


def jacobi(diag: torch.Tensor):
    """Jacobi preconditioner 1/diag(H) (bigwham4py.py:373-380)."""
    inv = 1.0 / diag
    return lambda v: inv * v


def warm_up(hmat, b: torch.Tensor, restart: int = 30) -> None:
    """One short restart cycle per precision, so that library initialisation
    (rocBLAS handles for the Gram-Schmidt products) is not timed."""
    for prec in hmat.precisions:
        gmres(lambda v: hmat.matvec(v, original=True, precision=prec), b, None,
              tol=0.0, restart=restart, maxiter=2)
    torch.cuda.synchronize()


def solve_fp64(hmat, b: torch.Tensor, tol: float = 1e-8, restart: int = 30,
               maxiter: int = 2000, precondition: bool = True) -> tuple[torch.Tensor, SolveInfo]:
    """Plain FP64 GMRES on the FP64 H-matvec (the baseline path)."""
    d = torch.from_numpy(hmat.diagonal(original=True)).to(b.device)
    M = jacobi(d) if precondition else None
    n64 = [0]

    def mv(v):
        n64[0] += 1
        return hmat.matvec(v, original=True, precision="fp64")

    _sync(b)
    t0 = time.perf_counter()
    x, its, _ = gmres(mv, b, M, tol=tol, restart=restart, maxiter=maxiter)
    r = b - hmat.matvec(x, original=True, precision="fp64")
    rel = (torch.linalg.vector_norm(r) / torch.linalg.vector_norm(b)).item()
    _sync(b)
    dt = time.perf_counter() - t0
    return x, SolveInfo(rel <= tol, its, n64[0] + 1, 0, rel, dt)


def solve_mixed(hmat, b: torch.Tensor, tol: float = 1e-8, inner_tol: float = 1e-5,
                restart: int = 30, maxiter: int = 2000, max_refine: int = 500,
                precondition: bool = True) -> tuple[torch.Tensor, SolveInfo]:
    """Iterative refinement: FP64 residuals, FP32-factor inner GMRES.

    Each refinement step solves H d = r with restarted GMRES on the FP32-factor
    matvec (FP64 Arnoldi and vectors; restarts take the residual from the
    Arnoldi relation, no extra matvec) down to max(inner_tol, 0.5 tol /
    (||r||/||b||)) of its right-hand side, then recomputes the exact FP64
    residual r = b - H x.  The FP32 operator is accurate to ~1e-7, so each
    refinement can gain about inner_tol; two to three FP64 matvecs reach
    1e-8."""
    d = torch.from_numpy(hmat.diagonal(original=True)).to(b.device)
    M = jacobi(d) if precondition else None
    counts = {"fp64": 0, "fp32": 0}

    def mv32(v):
        counts["fp32"] += 1
        return hmat.matvec(v, original=True, precision="fp32")

    _sync(b)
    t0 = time.perf_counter()
    bnorm = torch.linalg.vector_norm(b).item()
    x = torch.zeros_like(b)
    r = b.clone()
    rel = 1.0
    hist = []
    its = 0
    for _ in range(max_refine):
        target = max(inner_tol, 0.5 * tol / rel)
        dx, k, _ = gmres(mv32, r, M, tol=target, restart=restart, maxiter=maxiter - its,
                         implicit_restart=True)
        its += k
        x = x + dx
        r = b - hmat.matvec(x, original=True, precision="fp64")
        counts["fp64"] += 1
        rel = torch.linalg.vector_norm(r).item() / bnorm
        hist.append(rel)
        if rel <= tol or its >= maxiter:
            break
    _sync(b)
    dt = time.perf_counter() - t0
    return x, SolveInfo(rel <= tol, its, counts["fp64"], counts["fp32"], rel, dt, hist)
