"""bw_hip_matvec_noalloc on operators whose passes have more than 1 024 work
items and split slabs (a reduction launch adds the partial sums and there are no
counters to clear): the bits of bw_hip_matvec, in both precisions and
orderings, with a small operator that has counters called in between."""
import ctypes as C

import numpy as np
import pytest

from bigwham_dev_amd import HipHmat, HostHmat, set_tuning
from bigwham_dev_amd import _native as N
from bigwham_dev_amd.meshes import rect_grid
from synthetic_hmat import SyntheticHmat

pytestmark = pytest.mark.gpu


def _square(n):
    h = HostHmat.from_mesh("3DR0-H", *rect_grid(n), [1.0, 0.25])
    h.build(64, 3.0, 1e-6)
    return HipHmat(h, precisions=("fp64", "fp32"))


def _tuned():
    set_tuning(512, 512)
    try:
        return HipHmat(SyntheticHmat(400, 380, 2, 7), precisions=("fp64", "fp32"))
    finally:
        set_tuning(0, 0)


@pytest.mark.parametrize("make", [lambda: _square(64), _tuned], ids=["12288-dof", "tuned"])
def test_long_passes(gpu, make):
    import torch
    long, small = make(), _square(24)
    rng = np.random.default_rng(4)
    for precision, prec in (("fp64", N.BW_PREC_FP64), ("fp32", N.BW_PREC_FP32)):
        for original in (True, False, True):
            for dev in (long, small):
                print(f"noalloc {precision} original {original} rows {dev.n_rows}", flush=True)
                x = torch.from_numpy(rng.uniform(-1, 1, dev.n_cols)).to(gpu)
                y = torch.full((dev.n_rows,), np.nan, dtype=torch.float64, device=gpu)
                rc = N.hip().bw_hip_matvec_noalloc(
                    dev._h, C.c_void_p(x.data_ptr()), C.c_void_p(y.data_ptr()),
                    N.BW_ORDER_ORIGINAL if original else N.BW_ORDER_PERMUTED, prec,
                    C.c_void_p(torch.cuda.current_stream(gpu).cuda_stream))
                assert rc == N.BW_OK, N.hip().bw_hip_last_error().decode()
                assert torch.equal(y, dev.matvec(x, original=original, precision=precision))
    torch.cuda.synchronize()
