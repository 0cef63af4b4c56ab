"""The work-item lists of the slab layout, as the kernels take them (host only)."""
import ctypes as C

import numpy as np
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
        S = SyntheticHmat(*shape)  # owns what its flat() points to
        for info in _items_info(S.flat(), precision, False, wi).values():
            nwi, nred, _, counters, _ = info
            assert counters == (nred if nwi <= 1024 else 0), info
            few += nred > 0 and nwi <= 1024
            many += nred > 0 and nwi > 1024
    assert few and many  # both kinds were met


class Lists:
    """One direction's layout at one precision: data (in double), column groups, row
    map and the three work-item lists of both passes."""

    def __init__(self, flat, precision, adjoint, wi_bytes):
        lib, out = N.hip(), C.c_void_p()
        i64 = lambda a: a.ctypes.data_as(C.POINTER(C.c_int64))
        i32 = lambda a: a.ctypes.data_as(C.POINTER(C.c_int32))
        prec = N.BW_PREC_FP64 if precision == "fp64" else N.BW_PREC_FP32
        assert lib.bw_layout_build(C.byref(flat), prec, int(adjoint), wi_bytes,
                                   C.byref(out)) == N.BW_OK
        info = np.zeros(16, dtype=np.int64)
        lib.bw_layout_info(out, i64(info))
        self.xt_t, self.xt_size, self.V = int(info[0]), int(info[1]), int(info[14])
        self.rowmap = np.zeros(int(info[15]), dtype=np.int32)
        if self.rowmap.size:
            lib.bw_layout_export_rowmap(out, i32(self.rowmap))
        self.data, self.gidx, self.lists, self.rowtab = {}, {}, {}, None
        for p in (1, 2):
            gidx = np.zeros(max(1, int(info[3 + 6 * (p - 1)])), dtype=np.int32)
            data = np.zeros(int(info[5 + 6 * (p - 1)]))
            lib.bw_layout_export(out, p, None, i32(gidx), None,
                                 data.ctypes.data_as(C.POINTER(C.c_double)))
            self.gidx[p] = gidx[:int(info[3 + 6 * (p - 1)])].astype(np.int64)
            self.data[p] = data.reshape(-1, self.V)
            for k in range(3):
                n = np.zeros(5, dtype=np.int64)
                assert lib.bw_layout_items_info(out, p, k, i64(n)) == N.BW_OK
                wis = np.zeros((max(1, n[0]), 8), dtype=np.int64)
                reds = np.zeros((max(1, n[1]), 4), dtype=np.int64)
                xcd = np.zeros(9, dtype=np.int32)
                tab = np.zeros(self.rowmap.size, dtype=np.int64) if (p, k) == (1, 2) and n[0] else None
                assert lib.bw_layout_items_export(out, p, k, i64(wis), i64(reds), i32(xcd),
                                                  None if tab is None else i64(tab)) == N.BW_OK
                if tab is not None:
                    self.rowtab = tab
                self.lists[p, k] = dict(wis=wis[:n[0]], reds=reds[:n[1]], npart=int(n[2]),
                                        xcd=xcd, blocks=int(n[4]))
        lib.bw_layout_free(out)

    def vectors(self, p, k, wi):
        """(row, group) -> 16-byte vector of the pass's data, as the kernels form it:
        slabs group by group, windows through the row table with 32-bit offsets
        from the window's first row and 24-bit products."""
        doff, _, ng, R, orow = (int(v) for v in wi[:5])
        g = np.arange(ng)
        if k < 2:
            assert doff % self.V == 0
            return doff // self.V + g[None, :] * R + np.arange(R)[:, None]
        tab = self.rowtab[orow:orow + R]
        first = tab[0] >> 8
        stride = (tab & 0xff)[:, None]
        at = ((tab >> 8) - first)[:, None] + doff * stride
        assert at.min() >= 0 and doff + ng < 1 << 23 and stride.max() <= 64
        rel = at + g[None, :] * stride
        assert rel.max() < 1 << 31
        return first + rel


def _check_list(L, p, k):
    """Bounds, single coverage and the sums of split slabs of one list; returns the
    input group and the output row that it gives every vector."""
    W, l = 4, L.lists[p, k]
    nvec = L.data[p].shape[0]
    zin, out = np.full(nvec, -1), np.full(nvec, -1)
    n_rows = L.rowmap.size if p == 1 else None
    parts = np.zeros(l["npart"], dtype=int)
    by_red = {}
    for wi in l["wis"]:
        doff, gbeg, ng, R, orow, poff, red, _ = (int(v) for v in wi)
        assert 1 <= R <= 64 and ng >= 1 and gbeg >= 0 and gbeg + ng <= L.gidx[p].size
        z = L.gidx[p][gbeg:gbeg + ng]
        assert z.min() >= 0 and z.max() + L.V <= L.xt_size
        assert orow >= 0 and (n_rows is None or orow + R <= n_rows)
        at = L.vectors(p, k, wi)
        assert at.min() >= 0 and at.max() < nvec
        assert np.all(zin[at] == -1)
        zin[at] = z[None, :]
        out[at] = orow + np.arange(R)[:, None]
        # the waves' shares of the groups: contiguous, all of them, once
        nst = (ng + 3) // 4
        cuts = [min(ng, 4 * (nst * w // W)) for w in range(W + 1)]
        assert cuts[0] == 0 and cuts[-1] == ng and cuts == sorted(cuts)
        if poff >= 0:
            assert poff + R <= l["npart"] and red < len(l["reds"])
            parts[poff:poff + R] += 1
            by_red.setdefault(red, []).append((gbeg, poff, orow, R))
    assert np.all(zin >= 0) and np.all(parts == 1)
    assert sorted(by_red) == list(range(len(l["reds"])))
    for red, items in by_red.items():
        orow, R, poff, nparts = (int(v) for v in l["reds"][red])
        assert nparts == len(items) > 1
        for q, it in enumerate(sorted(items)):
            assert it[1:] == (poff + q * R, orow, R)
    # the launch: workgroup b takes item xcd[b % 8] + b / 8 of its XCD's range
    seen = np.zeros(len(l["wis"]), dtype=int)
    xs = l["xcd"]
    assert xs[0] == 0 and xs[-1] == len(l["wis"]) and np.all(np.diff(xs) >= 0)
    for b in range(l["blocks"]):
        w = xs[b % 8] + b // 8
        if w < xs[b % 8 + 1]:
            seen[w] += 1
    assert np.all(seen == 1)
    return zin, out


def _check_and_replay(S, precision, adjoint, wi_bytes):
    L = Lists(S.flat(), precision, adjoint, wi_bytes)
    d = S.dof
    n_in, n_out = (d * S.n_row_pts, d * S.n_col_pts) if adjoint else (d * S.n_col_pts, d * S.n_row_pts)
    x = np.random.default_rng(5).uniform(-1, 1, n_in)
    maps = {(p, k): _check_list(L, p, k) for p, k in L.lists if len(L.lists[p, k]["wis"])}
    for p in (1, 2):  # every list hands out the same products
        for k in (1, 2):
            if (p, k) in maps:
                assert all(np.array_equal(a, b) for a, b in zip(maps[p, 0], maps[p, k]))
    xt = np.zeros(L.xt_size)
    xt[:n_in] = x
    y = np.zeros(n_out)
    for p in (1, 2):
        if (p, 0) not in maps:
            continue
        zin, out = maps[p, 0]
        prod = (L.data[p] * xt[zin[:, None] + np.arange(L.V)]).sum(1)
        s = np.bincount(out, prod, minlength=L.rowmap.size if p == 1 else n_out)
        if p == 1:
            xt[L.rowmap] = s
        else:
            y += s
    blocks = [(q, (F,)) for q, F in zip(S.fr_pattern, S.fr)]
    blocks += [(q, (A, B)) for q, A, B in zip(S.lr_pattern, S.A, S.B)]
    ref, size = np.zeros(n_out), np.zeros(n_out)
    for (_, i0, j0, i1, j1, _), fs in blocks:
        rows, cols = slice(d * i0, d * i1), slice(d * j0, d * j1)
        if adjoint:
            rows, cols, fs = cols, rows, tuple(f.T for f in reversed(fs))
        v, b = x[cols], np.abs(x[cols])
        for f in reversed(fs):
            v, b = f @ v, np.abs(f) @ b
        ref[rows] += v
        size[rows] += b
    terms = n_in + int(S.lr_pattern[:, 5].sum())
    assert np.all(np.abs(y - ref) <= 4 * terms * 2.0 ** -53 * size)
    return set(maps)


@pytest.mark.parametrize("wi_bytes", [0, 512, 4096])
@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("shape", [(120, 90, 1, 1), (95, 140, 2, 2), (64, 200, 3, 3), (1, 75, 1, 4)])
def test_lists(shape, precision, adjoint, wi_bytes):
    _check_and_replay(SyntheticHmat(*shape), precision, adjoint, wi_bytes)


@pytest.mark.parametrize("adjoint", [False, True])
def test_windows(adjoint):
    """Long FP32 operators have windows over the slabs of a column cluster, which
    hand out the same products as the slabs."""
    S = SyntheticHmat(2300, 2400, 3, 12)
    assert (1, 2) in _check_and_replay(S, "fp32", adjoint, 0)
