"""The device orthogonalisation step (bw_hip_orthogonalize) against the same
classical Gram-Schmidt with re-orthogonalisation in numpy's longdouble: vector
lengths around the chunks and wave widths, one to many basis vectors.

Tolerances: the projected vector carries at most (n + 2k) u relative error per
pass, and the basis is orthonormal to the same order, so coefficients, norm and
next vector agree within 8 (n + 2k) u of ||w||."""
import ctypes as C

import numpy as np
import pytest

from bigwham_dev_amd import _native as N
from bigwham_dev_amd import solvers

pytestmark = pytest.mark.gpu
U = 2.0 ** -53


@pytest.mark.parametrize("n", [1, 63, 64, 255, 256, 257, 1000, 131072, 140001])
@pytest.mark.parametrize("k", [1, 7, 8, 9, 31])
def test_orthogonalize(gpu, n, k):
    import torch
    if k >= n and n > 1 or (n == 1 and k > 1):
        pytest.skip("no room for the next vector")
    print(f"orthogonalize n={n} k={k}", flush=True)
    rng = np.random.default_rng(n + k)
    Q = np.linalg.qr(rng.standard_normal((n, k)))[0].T.copy()
    w = rng.standard_normal(n)
    need = C.c_int64()
    assert N.hip().bw_hip_orthogonalize_work(n, k, C.byref(need)) == N.BW_OK
    V = torch.empty((k + 1, n), dtype=torch.float64, device=gpu)
    V[:k] = torch.from_numpy(Q).to(gpu)
    wd = torch.from_numpy(w).to(gpu)
    work = torch.full((need.value,), np.nan, dtype=torch.float64, device=gpu)
    col = torch.empty(k + 1, dtype=torch.float64, device=gpu)
    st = torch.cuda.current_stream(gpu).cuda_stream
    rc = N.hip().bw_hip_orthogonalize(V.device.index, n, k, V.data_ptr(), n, wd.data_ptr(),
                                      V[k].data_ptr(), col.data_ptr(), work.data_ptr(),
                                      need.value, st)
    assert rc == N.BW_OK
    L = np.longdouble
    Ql, wl = Q.astype(L), w.astype(L)
    h1 = Ql @ wl
    u = wl - Ql.T @ h1
    h2 = Ql @ u
    u = u - Ql.T @ h2
    hn = np.sqrt(u @ u)
    tol = 8 * (n + 2 * k) * U * float(np.linalg.norm(w))
    c = col.cpu().numpy()
    assert np.all(np.abs(c[:k] - (h1 + h2)) <= tol)
    assert abs(c[k] - hn) <= tol
    assert torch.equal(wd.cpu(), torch.from_numpy(w))  # w is left as it is
    if hn > 1e3 * tol:
        assert np.all(np.abs(V[k].cpu().numpy() - u / hn) <= 4 * tol / float(hn))


def test_arguments(gpu):
    lib = N.hip()
    need = C.c_int64()
    assert lib.bw_hip_orthogonalize_work(100, 1025, C.byref(need)) == N.BW_ESHAPE
    assert lib.bw_hip_orthogonalize_work(0, 3, C.byref(need)) == N.BW_EINVAL
    assert lib.bw_hip_orthogonalize_work(100, 3, C.byref(need)) == N.BW_OK
    assert lib.bw_hip_orthogonalize(0, 100, 3, 8, 100, 8, 8, 8, 8, need.value - 1, None) == N.BW_ESHAPE
    assert lib.bw_hip_orthogonalize(0, 100, 3, 8, 99, 8, 8, 8, 8, need.value, None) == N.BW_EINVAL


def test_operator_returning_its_input(gpu):
    """An identity operator hands back the basis vector itself: the step must
    not write to it, and the solve breaks down after one iteration."""
    import torch
    b = torch.arange(1.0, 51.0, dtype=torch.float64, device=gpu)
    x, its, rel = solvers.gmres(lambda v: v, b, restart=10, tol=1e-14)
    assert its <= 2 and torch.allclose(x, b, rtol=1e-13, atol=0)


@pytest.mark.parametrize("restart", [3, 12])
def test_strided_results(gpu, restart):
    """Operators whose result is not a contiguous float64 vector take the torch
    step; the solution is the same."""
    import torch
    rng = np.random.default_rng(3)
    A = torch.from_numpy(np.eye(80) * 2 + rng.standard_normal((80, 80)) / 9).to(gpu)
    b = torch.from_numpy(rng.standard_normal(80)).to(gpu)
    x0, _, r0 = solvers.gmres(lambda v: A @ v, b, restart=restart, tol=1e-11)
    x1, _, r1 = solvers.gmres(lambda v: torch.stack([A @ v, v], 1)[:, 0], b, restart=restart,
                              tol=1e-11)
    xe = torch.linalg.solve(A.cpu(), b.cpu())
    for x, r in ((x0, r0), (x1, r1)):
        assert r <= 1e-11
        assert torch.linalg.vector_norm(x.cpu() - xe) <= 1e-9 * torch.linalg.vector_norm(xe)
