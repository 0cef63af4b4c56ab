"""The work-item lists of the slab layout, as the kernels take them (host only)."""
import ctypes as C

import pytest

from bigwham_dev_amd import _native as N
from synthetic_hmat import SyntheticHmat


def _items_info(flat, precision, adjoint, wi_bytes):
    """{(pass, list): (work items, split slabs, partial sums, counters, workgroups)}"""
    lib, out = N.hip(), C.c_void_p()
    prec = N.BW_PREC_FP64 if precision == "fp64" else N.BW_PREC_FP32
    assert lib.bw_layout_build(C.byref(flat), prec, int(adjoint), wi_bytes, C.byref(out)) == N.BW_OK
    res = {}
    for p in (1, 2):
        for k in (0, 1, 2):
            info = (C.c_int64 * 5)()
            assert lib.bw_layout_items_info(out, p, k, info) == N.BW_OK
            res[p, k] = tuple(info)
    assert lib.bw_layout_items_info(out, 3, 0, (C.c_int64 * 5)()) == N.BW_EINVAL
    assert lib.bw_layout_items_info(out, 1, 3, (C.c_int64 * 5)()) == N.BW_EINVAL
    lib.bw_layout_free(out)
    return res


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_counters(precision):
    """A split slab has a counter in lists of at most 1 024 work items; longer
    lists have none at all, so that nothing clears or counts through a counter
    array that is not there."""
    few = many = 0
    for shape, wi in (((400, 380, 2, 7), 512), ((400, 380, 2, 7), 16384), ((95, 140, 2, 2), 0)):
        for info in _items_info(SyntheticHmat(*shape).flat(), precision, False, wi).values():
            nwi, nred, _, counters, _ = info
            assert counters == (nred if nwi <= 1024 else 0), info
            few += nred > 0 and nwi <= 1024
            many += nred > 0 and nwi > 1024
    assert few and many  # both kinds were met
