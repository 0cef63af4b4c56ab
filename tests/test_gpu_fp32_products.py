"""FP32 rounds of 16, 32 and 64 columns: every product has the accuracy of an FP32
multiplication, whatever sizes its row and column hold beside it, and large,
tiny and infinite numbers stay with the rows and columns that they belong to."""
import numpy as np
import pytest

from bigwham_dev_amd import HipHmat
from synthetic_hmat import SyntheticHmat

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _floats(rng, shape, lo, hi):
    """Floats of random sign and of sizes spread evenly over 2^lo .. 2^hi."""
    x = np.exp2(rng.uniform(lo, hi, shape)) * rng.choice([-1.0, 1.0], shape)
    return x.astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("cols", [10, 20, 40])
@pytest.mark.parametrize("a_range, x_range", [((-1, 1), (-1, 1)), ((-140, 20), (-60, 20)),
                                              ((-30, 90), (-120, -12)), ((-60, 20), (-140, 20))])
def test_single_products(gpu, cols, a_range, x_range):
    """Columns of X with one entry each, on full blocks: every result is one
    product, rounded once to the nearest float (half the smallest subnormal where
    the result is one); the additions of zeros round nothing."""
    import torch
    S = SyntheticHmat(130, 150, 2, 9, p_full=1.0)
    rng = np.random.default_rng(14)
    H = np.zeros((2 * 130, 2 * 150))
    for (_, i0, j0, i1, j1, _), F in zip(S.fr_pattern, S.fr):
        F[:] = _floats(rng, F.shape, *a_range)
        F[rng.random(F.shape) < 0.1] = 0.0
        H[2 * i0:2 * i1, 2 * j0:2 * j1] = F
    dev = HipHmat(S, precisions=("fp32",))
    at = rng.integers(0, 2 * 150, cols)
    X = np.zeros((2 * 150, cols))
    X[at, np.arange(cols)] = _floats(rng, cols, *x_range)
    Y = H[:, at] * X[at, np.arange(cols)]  # exact: 48 bits
    got = dev.matvec_batched(torch.from_numpy(X).to(gpu), original=False, precision="fp32")
    err = np.abs(got.cpu().numpy() - Y)
    assert np.all(err <= U * np.abs(Y) + 2.0 ** -150)


@pytest.mark.parametrize("adjoint", [False, True])
def test_windows_of_any_numbers(gpu, adjoint):
    """Pass 1 of 64-column rounds of long operators (windows over the slabs of a
    column cluster) with a column and an entry of large numbers, a column of tiny
    ones beside them, and an infinity."""
    import torch
    S = SyntheticHmat(2300, 2400, 3, 12)
    dev = HipHmat(S, precisions=("fp32",), adjoint=True)
    n_in = dev.n_rows if adjoint else dev.n_cols
    rng = np.random.default_rng(15)
    X = rng.uniform(-1, 1, (n_in, 64))
    X[:, 5] *= 1e-33
    blocks = [(p, (F,)) for p, F in zip(S.fr_pattern, S.fr)]
    blocks += [(p, (A, B)) for p, A, B in zip(S.lr_pattern, S.A, S.B)]
    n_out = dev.n_cols if adjoint else dev.n_rows
    for case in ("column", "entry"):
        if case == "column":
            Z = X.copy()
            Z[:, 3] *= 1e30
        else:
            Z = X.copy()
            Z[n_in // 3, 7] = 1e33
        Y, bound = np.zeros((n_out, 64)), np.zeros((n_out, 64))
        for (_, i0, j0, i1, j1, _), fs in blocks:
            rows, cols = slice(3 * i0, 3 * i1), slice(3 * j0, 3 * j1)
            if adjoint:
                rows, cols, fs = cols, rows, tuple(f.T for f in reversed(fs))
            v, b = Z[cols], np.abs(Z[cols])
            for f in reversed(fs):
                v, b = f @ v, np.abs(f) @ b
            Y[rows] += v
            bound[rows] += b
        tol = 2 * (n_in + int(S.lr_pattern[:, 5].sum()) + 8) * U * bound
        print(f"windows, {case}, adjoint {adjoint}", flush=True)
        got = dev.matvec_batched(torch.from_numpy(Z).to(gpu), original=False, precision="fp32",
                                 adjoint=adjoint)
        assert np.all(np.abs(got.cpu().numpy() - Y) <= tol), case
    X[n_in // 2, 9] = np.inf
    Xd = torch.from_numpy(X).to(gpu)
    got = dev.matvec_batched(Xd, original=False, precision="fp32", adjoint=adjoint).cpu().numpy()
    for j in (8, 9, 10):
        y = dev.matvec(Xd[:, j].contiguous(), original=False, precision="fp32",
                       adjoint=adjoint).cpu().numpy()
        assert np.array_equal(np.isnan(got[:, j]), np.isnan(y)), j
        assert np.array_equal(np.isposinf(got[:, j]), np.isposinf(y)), j
        assert np.array_equal(np.isneginf(got[:, j]), np.isneginf(y)), j
    assert np.all(np.isfinite(np.delete(got, 9, axis=1)))
