"""What operators and right-hand sides the device GMRES takes and refuses is what
the same solve takes and refuses on the CPU, where every step is torch's:
differentiation through the step is refused, and results that cannot be read
through a pointer are solved like any other."""
import pytest
import torch
from torch.autograd import forward_ad

from bigwham_dev_amd.solvers import _DeviceSteps, gmres

pytestmark = pytest.mark.gpu


class Sub(torch.Tensor):
    pass


def _system(device):
    g = torch.Generator().manual_seed(3)
    A = torch.eye(40, dtype=torch.float64) * 3
    A = A + torch.randn(40, 40, generator=g, dtype=torch.float64) / 9
    b = torch.randn(40, generator=g, dtype=torch.float64)
    return A.to(device), b.to(device)


def _dual(f):
    def call(A, b):
        with forward_ad.dual_level():
            return f(A, b)
    return call


REFUSED = {
    "operator with a gradient": lambda A, b: gmres(lambda v: A.requires_grad_(True) @ v, b),
    "right-hand side with a gradient": lambda A, b: gmres(lambda v: A @ v, b.requires_grad_(True)),
    "detached operator": lambda A, b: gmres(lambda v: A @ v.detach(), b.requires_grad_(True)),
    "operator with a tangent": _dual(lambda A, b: gmres(
        lambda v: forward_ad.make_dual(A, torch.ones_like(A)) @ v, b)),
    "right-hand side with a tangent": _dual(lambda A, b: gmres(
        lambda v: A @ v, forward_ad.make_dual(b, torch.ones_like(b)))),
    "func.grad": lambda A, b: torch.func.grad(lambda c: gmres(lambda v: A @ v, c)[0].sum())(b),
    "func.jvp": lambda A, b: torch.func.jvp(lambda c: gmres(lambda v: A @ v, c)[0], (b,), (b,)),
    "vmap": lambda A, b: torch.func.vmap(lambda c: gmres(lambda v: A @ v, c)[0])(
        torch.stack([b, b])),
}

TAKEN = {
    "plain": lambda A, b: gmres(lambda v: A @ v, b, tol=1e-11),
    "gradients off": lambda A, b: torch.no_grad()(gmres)(
        lambda v: A.requires_grad_(True) @ v, b, tol=1e-11),
    "inference mode": lambda A, b: torch.inference_mode()(gmres)(lambda v: A @ v, b, tol=1e-11),
    "negated view": lambda A, b: gmres(lambda v: torch._neg_view(-(A @ v)), b, tol=1e-11),
    "subclass": lambda A, b: gmres(lambda v: (A @ v).as_subclass(Sub), b, tol=1e-11),
}


@pytest.mark.parametrize("name", list(REFUSED))
def test_refused(gpu, name):
    errors = []
    for device in ("cpu", gpu):
        with pytest.raises((RuntimeError, NotImplementedError)) as e:
            REFUSED[name](*_system(device))
        errors.append(type(e.value))
    assert errors[0] is errors[1]


@pytest.mark.parametrize("name", list(TAKEN))
def test_taken(gpu, name):
    A, b = _system("cpu")
    exact = torch.linalg.solve(A, b)
    x, _, rel = TAKEN[name](*_system(gpu))
    assert rel <= 1e-11 and not x.requires_grad
    # ||x - exact|| <= ||A^-1|| tol ||b||, and the smallest singular value of A is above 1
    assert torch.linalg.svdvals(A).min() > 1
    assert torch.linalg.vector_norm(x.cpu() - exact) <= 2e-11 * torch.linalg.vector_norm(b)


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two GPUs")
def test_current_device_is_kept(gpu):
    """A solve on the second GPU leaves the first one current, as torch does."""
    A, b = _system("cuda:1")
    with torch.cuda.device(0):
        _, _, rel = gmres(lambda v: A @ v, b, tol=1e-11)
        assert rel <= 1e-11
        assert torch.empty(1, device="cuda").device.index == 0


def test_pinned_columns(gpu):
    """The pinned memory of a solve grows with the restart length, not with its
    square (a full-memory solve restarts after thousands of vectors)."""
    steps = _DeviceSteps(torch.empty((3001, 8), dtype=torch.float64, device=gpu))
    assert steps.cols.is_pinned() and steps.cols.numel() <= 4 * 3001
    steps.close()


@pytest.mark.parametrize("strided", [False, True])
@pytest.mark.parametrize("restart", [1, 2, 3, 39])
def test_restarts(gpu, restart, strided):
    """Cycles of one step up to the whole space, through the native and the torch
    step: as many iterations as on the CPU, give or take the last bits."""
    op = lambda A: lambda v: torch.stack([A @ v, v], 1)[:, 0] if strided else A @ v
    A, b = _system("cpu")
    _, n, _ = gmres(op(A), b, restart=restart, tol=1e-10)
    A, b = _system(gpu)
    x, m, rel = gmres(op(A), b, restart=restart, tol=1e-10)
    assert rel <= 1e-10 and abs(m - n) <= 1
    # the residual itself: rounding of a 40-term product is far below the tolerance
    assert torch.linalg.vector_norm(b - A @ x) <= 1.01e-10 * torch.linalg.vector_norm(b)
