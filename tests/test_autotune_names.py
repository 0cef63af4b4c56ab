"""The names of the autotuner that programs loop over: its lists of unroll depths,
batched schedules and work-item sizes hold only values that the engine takes,
and tune_mfma times every schedule of its list."""
import pytest

from bigwham_dev_amd import autotune


def test_lists():
    assert set(autotune.UNROLLS) <= {4, 8, 16}
    for schedules in (autotune.MFMA_SCHEDULES, autotune.MFMA64_SCHEDULES):
        assert len(schedules) >= 1 and all(0 <= s <= 15 for s in schedules)
    assert all(b > 0 for b in autotune.WI_BYTES)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_tune_mfma(gpu, precision):
    from bigwham_dev_amd import HipHmat
    from synthetic_hmat import SyntheticHmat
    dev = HipHmat(SyntheticHmat(95, 140, 2, 2), precisions=(precision,))
    schedules = autotune.MFMA_SCHEDULES if precision == "fp32" else autotune.MFMA64_SCHEDULES
    r = autotune.tune_mfma(dev, nrhs=20, reps=2, precision=precision)
    assert set(r) == set(schedules) | {"best"} and r["best"] in schedules
    assert all(r[s] > 0 for s in schedules)
