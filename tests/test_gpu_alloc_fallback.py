"""Allocation failures that a call handles: FP32 batched scratch that does not fit
64 columns wide is made 32 wide and the call succeeds, and after a call that
returned BW_ENOMEM the next ones work.  With BWHIP_FAIL_ALLOC_AT=k the k-th
allocation of a call fails in the runtime itself, which then has an error
pending that later launch checks would report."""
import ctypes as C

import numpy as np
import pytest

from bigwham_dev_amd import HipHmat, set_tuning
from bigwham_dev_amd import _native as N
from synthetic_hmat import SyntheticHmat

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def case(gpu):
    import torch
    S = SyntheticHmat(95, 140, 2, 2)
    X = torch.from_numpy(np.random.default_rng(1).uniform(-1, 1, (2 * 140, 40))).to(gpu)
    dev = HipHmat(S, precisions=("fp32",))
    # rounds of 32 and 16 columns, which a 32-wide scratch takes for these 40
    Y = torch.cat([dev.matvec_batched(X[:, k:k + 32], precision="fp32") for k in (0, 32)], 1)
    return S, X, Y


@pytest.mark.parametrize("k", [1, 2, 3])
def test_narrow_scratch(case, gpu, monkeypatch, k):
    import torch
    S, X, Y = case
    dev = HipHmat(S, precisions=("fp32",))
    monkeypatch.setenv("BWHIP_FAIL_ALLOC_AT", str(k))
    print(f"batched scratch, allocation {k} failing", flush=True)
    got = dev.matvec_batched(X, precision="fp32")
    monkeypatch.delenv("BWHIP_FAIL_ALLOC_AT")
    assert torch.equal(got, Y)
    assert torch.equal(dev.matvec_batched(X, precision="fp32"), Y)


@pytest.mark.parametrize("k", [4, 5, 6])  # after the three of the single-vector scratch
def test_narrow_scratch_of_a_graph(case, gpu, monkeypatch, k):
    import torch
    S, X, Y = case
    dev = HipHmat(S, precisions=("fp32",))
    monkeypatch.setenv("BWHIP_FAIL_ALLOC_AT", str(k))
    print(f"graph scratch, allocation {k} failing", flush=True)
    g = dev.graph_batched(X, precision="fp32")
    monkeypatch.delenv("BWHIP_FAIL_ALLOC_AT")
    for _ in range(3):
        assert torch.equal(g.launch(), Y)
        torch.cuda.synchronize()


@pytest.mark.parametrize("host", [False, True])
def test_call_after_a_failed_one(case, gpu, monkeypatch, host):
    """The failed call leaves no error behind: not for the same handle, not for
    torch on the same thread."""
    import torch
    S, X, _ = case
    dev = HipHmat(S, precisions=("fp32",))
    x = X[:, 0].contiguous()
    ref = dev.matvec(x, precision="fp32")
    s = torch.cuda.Stream(gpu)
    hx, hy = x.cpu().numpy(), np.empty(dev.n_rows)
    y = torch.empty_like(ref)
    for k in (1, 2, 3, 4, 5) if host else (1, 2, 3):
        monkeypatch.setenv("BWHIP_FAIL_ALLOC_AT", str(k))
        print(f"host {host}, allocation {k} failing", flush=True)
        px, py = (hx.ctypes.data, hy.ctypes.data) if host else (x.data_ptr(), y.data_ptr())
        rc = N.hip().bw_hip_matvec(dev._h, C.c_void_p(px), C.c_void_p(py), N.BW_ORDER_ORIGINAL,
                                   N.BW_PREC_FP32, 0 if host else 1, C.c_void_p(s.cuda_stream))
        assert rc == N.BW_ENOMEM
        if host:
            # the single-vector scratch of an earlier try is kept
            N.check_hip(N.hip().bw_hip_stream_release(dev._h, C.c_void_p(s.cuda_stream)))
        monkeypatch.delenv("BWHIP_FAIL_ALLOC_AT")
        assert torch.equal(dev.matvec(x, precision="fp32"), ref)
        assert torch.equal((x + x) - x, x)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_failed_zero_fill(gpu, monkeypatch, precision):
    """A batched call that is the first on its stream makes both kinds of scratch;
    whichever of its zero fills fails, the calls that follow on that stream
    have scratch of their own or make it anew, and all of it is given back."""
    import torch
    set_tuning(16384, 16384)  # split slabs, so that there are counters to clear
    try:
        dev = HipHmat(SyntheticHmat(400, 380, 2, 7), precisions=(precision,))
    finally:
        set_tuning(0, 0)
    X = torch.from_numpy(np.random.default_rng(2).uniform(-1, 1, (dev.n_cols, 40))).to(gpu)
    x = X[:, 0].contiguous()
    Y, y = dev.matvec_batched(X, precision=precision), dev.matvec(x, precision=precision)
    s = torch.cuda.Stream(gpu)
    with torch.cuda.stream(s):
        torch.zeros(1, device=gpu)
        Ys, ys = torch.empty_like(Y), torch.empty_like(y)
    failed = 0
    for k in range(20):  # 0: none, so that torch's own buffers are there
        monkeypatch.setenv("BWHIP_FAIL_FILL_AT", str(k))
        print(f"{precision}, zero fill {k} failing", flush=True)
        with torch.cuda.stream(s):
            try:
                dev.matvec_batched(X, precision=precision, out=Ys)
                ok = True
            except N.BigWhamError as e:
                assert "zero fill" in str(e)
                ok = False
            monkeypatch.delenv("BWHIP_FAIL_FILL_AT")
            dev.matvec(x, precision=precision, out=ys)
            assert torch.equal(ys, y)
            dev.matvec_batched(X, precision=precision, out=Ys)
            assert torch.equal(Ys, Y)
        dev.release_stream(s.cuda_stream)
        torch.cuda.synchronize()
        if k == 0:
            before = torch.cuda.mem_get_info(0)[0]
            continue
        assert torch.cuda.mem_get_info(0)[0] == before
        if ok:
            break
        failed += 1
    assert ok and failed >= 3  # xt, and counters of both kinds of scratch
