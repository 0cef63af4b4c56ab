"""Work items shared by the waves of a workgroup, at the sizes where the split
can go wrong: slabs of 1 to 64 rows (edges of the 16- and 32-row tiles), items
of fewer column groups than a workgroup has waves, remainders of every batch
depth, whole slabs and slabs split over several items; and rounds of every
width of the batched product (16, 32 and 64 columns and their edges) in any
order on one handle, against the operator's blocks multiplied in numpy.

The tolerance is the a-priori bound of a sum of products in the working
precision: |y - H x| <= n u (|F| |x| + |A| (|B| |x|)) with n the terms of the
longest row (columns plus total rank, twice for the two passes, plus the
conversion of factors and input), u the unit roundoff."""
import numpy as np
import pytest

from bigwham_dev_amd import HipHmat, set_tuning
from synthetic_hmat import SyntheticHmat

pytestmark = pytest.mark.gpu

U = {"fp64": 2.0 ** -53, "fp32": 2.0 ** -24}
# (row points, column points, dof, seed): slabs of many heights, few and many
# columns, one-row and one-column point sets
SHAPES = [(120, 90, 1, 1), (95, 140, 2, 2), (64, 200, 3, 3), (1, 75, 1, 4), (75, 1, 3, 5)]


def _reference(S, X, adjoint):
    """H X (H^T X) in permuted order, and |F| |X| + |A| (|B| |X|)."""
    d = S.dof
    n_out = d * (S.n_col_pts if adjoint else S.n_row_pts)
    Y, B = np.zeros((n_out, X.shape[1])), np.zeros((n_out, X.shape[1]))
    blocks = [(p, (F,)) for p, F in zip(S.fr_pattern, S.fr)]
    blocks += [(p, (A, Bf)) for p, A, Bf in zip(S.lr_pattern, S.A, S.B)]
    for (_, i0, j0, i1, j1, _), fs in blocks:
        rows, cols = slice(d * i0, d * i1), slice(d * j0, d * j1)
        if adjoint:
            rows, cols, fs = cols, rows, tuple(f.T for f in reversed(fs))
        v, b = X[cols], np.abs(X[cols])
        for f in reversed(fs):
            v, b = f @ v, np.abs(f) @ b
        Y[rows] += v
        B[rows] += b
    return Y, B


@pytest.mark.parametrize("wi_bytes", [0, 512, 4096])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", SHAPES)
def test_single_and_batched(gpu, shape, precision, wi_bytes):
    import torch
    S = SyntheticHmat(*shape)
    set_tuning(wi_bytes, wi_bytes)
    try:
        dev = HipHmat(S, precisions=(precision,), adjoint=True)
    finally:
        set_tuning(0, 0)
    for adjoint in (False, True):
        n_in = dev.n_rows if adjoint else dev.n_cols
        print(f"work items {shape} {precision} wi {wi_bytes} adjoint {adjoint}", flush=True)
        X = np.random.default_rng(sum(shape)).uniform(-1, 1, (n_in, 32))
        Y, bound = _reference(S, X, adjoint)
        terms = n_in + int(S.lr_pattern[:, 5].sum()) + 8
        tol = 2 * terms * U[precision] * bound
        Xd = torch.from_numpy(X).to(gpu)
        got = dev.matvec_batched(Xd, original=False, precision=precision, adjoint=adjoint)
        assert np.all(np.abs(got.cpu().numpy() - Y) <= tol)
        for j in (0, 31):
            for u in (4, 8):
                dev.set_unroll(u, u)
                y = dev.matvec(Xd[:, j].contiguous(), original=False, precision=precision,
                               adjoint=adjoint)
                assert np.all(np.abs(y.cpu().numpy() - Y[:, j]) <= tol[:, j]), (j, u)
        # the same product in the original numbering, moved by both permutations
        p_in, p_out = (S.perm0, S.perm1) if adjoint else (S.perm1, S.perm0)
        dofs = np.arange(S.dof)
        x = np.empty(n_in)
        x[(S.dof * p_in[:, None] + dofs).ravel()] = X[:, 31]
        yo = dev.matvec(torch.from_numpy(x).to(gpu), original=True, precision=precision,
                        adjoint=adjoint).cpu().numpy()
        assert np.array_equal(yo[(S.dof * p_out[:, None] + dofs).ravel()], y.cpu().numpy())


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(95, 140, 2, 2), (64, 200, 3, 3), (40, 33, 3, 6)])
def test_round_widths(gpu, shape, precision):
    """Column counts at the edges of the rounds, wide before narrow and back
    (the rounds share one scratch buffer), row- and column-major operands."""
    import torch
    S = SyntheticHmat(*shape)
    dev = HipHmat(S, precisions=(precision,))
    terms = dev.n_cols + int(S.lr_pattern[:, 5].sum()) + 8
    for k in (64, 1, 33, 16, 17, 48, 15, 65, 32, 100, 7):
        X = np.random.default_rng(k).uniform(-1, 1, (dev.n_cols, k))
        Y, bound = _reference(S, X, False)
        tol = 2 * terms * U[precision] * bound
        Xd = torch.from_numpy(X).to(gpu)
        Xc = torch.from_numpy(np.ascontiguousarray(X.T)).to(gpu).t()
        print(f"round widths {shape} {precision} k {k}", flush=True)
        got = dev.matvec_batched(Xd, original=False, precision=precision)
        assert np.all(np.abs(got.cpu().numpy() - Y) <= tol), k
        out = torch.full((k, dev.n_rows), np.nan, dtype=torch.float64, device=gpu).t()
        dev.matvec_batched(Xc, original=False, precision=precision, out=out)
        assert torch.equal(out, got), k


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("wi_bytes", [512, 4096])
def test_split_slabs(gpu, precision, wi_bytes):
    """Slabs split over several work items, in passes of few (the last item of
    a slab adds the partial sums) and of many work items (a reduction launch
    does): against the blocks, and the same bits on every launch, whatever
    order the items finish in: eager, on two streams at once and in a graph."""
    import torch
    S = SyntheticHmat(400, 380, 2, 7)
    set_tuning(wi_bytes, wi_bytes)
    try:
        dev = HipHmat(S, precisions=(precision,))
    finally:
        set_tuning(0, 0)
    X = np.random.default_rng(8).uniform(-1, 1, (dev.n_cols, 40))
    Y, bound = _reference(S, X, False)
    tol = 2 * (dev.n_cols + int(S.lr_pattern[:, 5].sum()) + 8) * U[precision] * bound
    Xd = torch.from_numpy(X).to(gpu)
    x = Xd[:, 0].contiguous()
    y = dev.matvec(x, original=False, precision=precision)
    Yd = dev.matvec_batched(Xd, original=False, precision=precision)
    assert np.all(np.abs(y.cpu().numpy() - Y[:, 0]) <= tol[:, 0])
    assert np.all(np.abs(Yd.cpu().numpy() - Y) <= tol)
    g = dev.graph(x, original=False, precision=precision)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    outs = []
    for rep in range(20):
        for s in streams:
            with torch.cuda.stream(s):
                outs.append((dev.matvec(x, original=False, precision=precision), y))
                outs.append((dev.matvec_batched(Xd, original=False, precision=precision), Yd))
        outs.append((g.launch().clone(), y))
    torch.cuda.synchronize()
    for a, b in outs:
        assert torch.equal(a, b)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(1024, 40, 1, 1), (1025, 40, 1, 2), (3, 131072, 1, 3),
                                   (3, 131073, 1, 4), (350, 342, 3, 5),
                                   (90, 2048, 3, 6), (90, 2049, 3, 7)])
def test_host_vectors(gpu, shape, precision):
    """Host vectors give the bits of device vectors, at the sizes where their
    way changes (1 024 results, 6 144 and 131 072 entries), repeated with new inputs (the
    staging is shared), in both orderings and directions."""
    import torch
    S = SyntheticHmat(*shape)
    dev = HipHmat(S, precisions=(precision,), adjoint=True)
    rng = np.random.default_rng(6)
    for adjoint in (False, True, False):
        for original in (True, False):
            x = rng.uniform(-1, 1, dev.n_rows if adjoint else dev.n_cols)
            y = dev.matvec(x, original=original, precision=precision, adjoint=adjoint)
            yd = dev.matvec(torch.from_numpy(x).to(gpu), original=original, precision=precision,
                            adjoint=adjoint)
            assert np.array_equal(y, yd.cpu().numpy()), (adjoint, original)


@pytest.mark.parametrize("cols", [20, 40])
@pytest.mark.parametrize("a_scale, x_scale", [
    (1.0, 1.0), (1.0, 1e-28), (1.0, 1e-33), (1.0, 1e30), (1e-22, 1e-12), (1e-22, 1e20)])
def test_fp32_split_range(gpu, cols, a_scale, x_scale):
    """The 32- and 64-wide FP32 rounds split their numbers into bf16 parts where
    that is exact: operators and inputs of sizes within, at the end of and
    outside that range, and columns of other sizes beside them.  Products
    below 2^-126 may be lost (the last term)."""
    import torch
    S = SyntheticHmat(130, 150, 2, 9)
    for blocks in (S.fr, S.A):
        for b in blocks:
            b *= a_scale
    dev = HipHmat(S, precisions=("fp32",))
    X = np.random.default_rng(10).uniform(-1, 1, (dev.n_cols, cols)) * x_scale
    X[:, 3] /= x_scale   # columns of ordinary size, of one tiny entry, of zeros
    X[5:, 4] = 0.0
    X[4, 4] = 3e-38
    X[:, 5] = 0.0
    Y, bound = _reference(S, X, False)
    n = dev.n_cols + int(S.lr_pattern[:, 5].sum()) + 8
    got = dev.matvec_batched(torch.from_numpy(X).to(gpu), original=False, precision="fp32")
    big = max(1.0, max(np.abs(b).sum(axis=1).max(initial=0.0) for b in S.fr + S.A))
    assert np.all(np.abs(got.cpu().numpy() - Y) <= 2 * n * U["fp32"] * bound + n * big * 2.0 ** -126)


@pytest.mark.parametrize("cols", [20, 40])
def test_fp32_not_finite(gpu, cols):
    """Infinities and NaN in the input of a wide FP32 round reach the entries
    that they reach in the single-vector product, and no other column."""
    import torch
    S = SyntheticHmat(130, 150, 2, 9)
    dev = HipHmat(S, precisions=("fp32",))
    X = np.random.default_rng(11).uniform(-1, 1, (dev.n_cols, cols))
    X[7, 2], X[90, 3], X[200, 4] = np.inf, -np.inf, np.nan
    Xd = torch.from_numpy(X).to(gpu)
    got = dev.matvec_batched(Xd, original=False, precision="fp32").cpu().numpy()
    for j in range(cols):
        y = dev.matvec(Xd[:, j].contiguous(), original=False, precision="fp32").cpu().numpy()
        assert np.array_equal(np.isnan(got[:, j]), np.isnan(y)), j
        assert np.array_equal(np.isposinf(got[:, j]), np.isposinf(y)), j
        assert np.array_equal(np.isneginf(got[:, j]), np.isneginf(y)), j
        assert j in (2, 3, 4) or np.all(np.isfinite(y))


@pytest.mark.parametrize("adjoint", [False, True])
def test_windows(gpu, adjoint):
    """Rounds of 64 columns of long FP32 operators take pass 1 in windows over
    the slabs of a column cluster: the same columns as narrower rounds give,
    within the bound, and the same bits on every launch."""
    import torch
    S = SyntheticHmat(2300, 2400, 3, 12)
    assert sum(b.size for b in S.B) > 13 << 20 and sum(a.size for a in S.A) > 13 << 20
    dev = HipHmat(S, precisions=("fp32",), adjoint=True)
    n_in = dev.n_rows if adjoint else dev.n_cols
    X = np.random.default_rng(13).uniform(-1, 1, (n_in, 100))
    Y, bound = _reference(S, X, adjoint)
    tol = 2 * (n_in + int(S.lr_pattern[:, 5].sum()) + 8) * U["fp32"] * bound
    Xd = torch.from_numpy(X).to(gpu)
    for cols in (33, 64, 100):
        y = dev.matvec_batched(Xd[:, :cols], original=False, precision="fp32", adjoint=adjoint)
        assert np.all(np.abs(y.cpu().numpy() - Y[:, :cols]) <= tol[:, :cols]), cols
        for _ in range(3):
            assert torch.equal(y, dev.matvec_batched(Xd[:, :cols], original=False,
                                                     precision="fp32", adjoint=adjoint))
    # 16 at a time: no windows; FP32 errors of the two ways only
    z = torch.cat([dev.matvec_batched(Xd[:, k:k + 16], original=False, precision="fp32",
                                      adjoint=adjoint) for k in range(0, 100, 16)], 1)
    assert torch.linalg.vector_norm(z - y) <= 1e-6 * torch.linalg.vector_norm(y)
