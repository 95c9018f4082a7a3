"""The packed single-workgroup tail of the coloured V-cycle (resident and streamed levels)
gives the bits of the launched cycle: sizes at the edges of its items (64 rows), of the
single-wavefront levels and of what stays resident; both precisions, one and two sweeps."""
import numpy as np
import pytest

import matgen
from test_gpu_parity import gpu_amg, ls_from

pytestmark = pytest.mark.gpu


def box_rows(n, seed):
    """A random sparse matrix without structure: non-symmetric pattern, ragged rows."""
    rng = np.random.default_rng(seed)
    row, col, off = [0], [], []
    for i in range(n):
        c = rng.choice(n, size=min(n - 1, int(rng.integers(0, 24))), replace=False)
        c = c[c != i]
        col += list(c)
        off += list(rng.uniform(0.01, 1.0, len(c)))
        row.append(len(col))
    diag = np.array([-1.2 * sum(off[row[i]:row[i + 1]]) - 0.1 for i in range(n)])
    return dict(n_self=n, n_total=n, row=np.array(row, np.int32), col=np.array(col, np.int32), diag=diag,
                off=np.array(off), b=rng.uniform(-1, 1, n))


CASES = {"chain65": lambda: matgen.chain(65, d=-2.1), "chain130": lambda: matgen.chain(130, d=-2.1),
         "grid5": lambda: matgen.grid3d(5, seed=1), "grid11": lambda: matgen.grid3d(11, seed=2, contrast=1.5),
         "grid21": lambda: matgen.grid3d(21, seed=3, contrast=2.0), "grid26": lambda: matgen.grid3d(26, seed=4),
         "ragged63": lambda: box_rows(63, 5), "ragged700": lambda: box_rows(700, 6),
         "ragged3000": lambda: box_rows(3000, 7)}


@pytest.mark.parametrize("prec,npost", [(0, 1), (1, 1), (0, 2), (1, 2)])
@pytest.mark.parametrize("case", sorted(CASES))
def test_packed_tail_is_bit_identical(case, prec, npost):
    m = CASES[case]()
    res = []
    for tail in (0, 6000, 1 << 30):
        a = gpu_amg(gsOrdering=1, precision=prec, nPostSweeps=npost, nMaxIterations=6, relativeTolerance=1e-30)
        a.set_tuning("tail_max_rows", tail)
        ls = ls_from(m)
        a.solve(ls)
        res.append((ls.delta.copy(), a.history()))
        # the packed form ran, from the first level that fits the limit, with levels streamed and resident
        form, first, resident = (a.get_tuning("tail_" + k) for k in ("form", "level", "resident_level"))
        n = [a.level(l)["n"] for l in range(a.num_levels())]
        assert form == (2 if tail else 0)
        assert first == (next(l for l in range(1, len(n)) if n[l] <= tail) if tail else -1)
        assert not tail or (resident > first if n[first] > 1000 else resident >= first)
    for d, h in res[1:]:
        assert np.array_equal(res[0][0], d) and np.array_equal(res[0][1], h)


FLOW = {"chain300": lambda: matgen.chain(300, d=-2.1), "grid4": lambda: matgen.grid3d(4, seed=1),
        "grid17": lambda: matgen.grid3d(17, seed=2, contrast=1.5), "grid24": lambda: matgen.grid3d(24, seed=3),
        "ragged63": lambda: box_rows(63, 5), "ragged700": lambda: box_rows(700, 6),
        "ragged3000": lambda: box_rows(3000, 7),
        # one dependency level of more than 64 rows, rows without entries, a deep chain behind
        "empty500": lambda: dict(matgen.chain(500), row=np.zeros(501, np.int32), col=np.zeros(0, np.int32),
                                 off=np.zeros(0))}


@pytest.mark.parametrize("prec,npost", [(0, 1), (1, 1), (0, 2)])
@pytest.mark.parametrize("case", sorted(FLOW))
def test_one_workgroup_reference_sweep_is_bit_identical(case, prec, npost):
    """Reference-order sweeps by one workgroup (every level of these is swept by it) and by the whole
    chip (exact_flow_wg_rows 0) against the level-by-level launches."""
    m = FLOW[case]()
    res = []
    for flow, wg_rows in ((0, 0), (1, 150000), (1, 0)):
        a = gpu_amg(gsOrdering=0, precision=prec, nPostSweeps=npost, nMaxIterations=6, relativeTolerance=1e-30)
        a.set_tuning("exact_flow", flow)
        a.set_tuning("exact_flow_wg_rows", wg_rows)
        ls = ls_from(m)
        a.solve(ls)
        res.append((ls.delta.copy(), a.history()))
        # an empty level is not swept at all
        swept = [l for l in range(a.num_levels()) if flow and 0 < a.level(l)["n"] <= wg_rows]
        assert a.get_tuning("exact_flow_wg_levels") == sum(1 << l for l in swept)
    for d, h in res[1:]:
        assert np.array_equal(res[0][0], d) and np.array_equal(res[0][1], h)


def bundle(n, hub, seed=0):
    """Rows in bundles of 64, each linked to the same row of the bundle before (a dependency level per
    bundle); the first row of every bundle reads ``hub`` rows of earlier bundles besides."""
    rng = np.random.default_rng(seed)
    rows = []
    for i in range(n):
        c = {j for j in (i - 64, i + 64) if 0 <= j < n}
        if hub and i % 64 == 0 and i > 64:
            c |= {int(j) for j in rng.integers(0, i - i % 64, hub)}
        rows.append(sorted(c))
    row = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    off = rng.uniform(0.1, 1.0, row[-1])
    diag = np.array([-1.1 * off[row[i]:row[i + 1]].sum() - 0.1 for i in range(n)])
    return dict(n_self=n, n_total=n, row=row, col=np.array([c for r in rows for c in r], np.int32), diag=diag,
                off=off, b=rng.uniform(-1, 1, n))


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("hub,used", [(0, True), (80, True), (300, False)])
def test_level_with_hub_rows_is_not_padded_to_them(prec, hub, used):
    """Items of one hub and 63 short rows: 64 rows padded to 300 entries each take nine groups of four
    per entry and row of the level (limit: eight; hubs of 80: 4.6), so the chip-wide sweep keeps it.
    Same bits either way."""
    m = bundle(2560, hub)
    res = []
    for flow in (0, 1):
        a = gpu_amg(gsOrdering=0, precision=prec, nMaxIterations=6, relativeTolerance=1e-30)
        a.set_tuning("exact_flow", flow)
        ls = ls_from(m)
        a.solve(ls)
        res.append((ls.delta.copy(), a.history()))
        assert a.get_tuning("exact_flow_wg_levels") & 1 == (flow and used)
    assert np.array_equal(res[0][0], res[1][0]) and np.array_equal(res[0][1], res[1][1])


def layered(n, dists, hub=0, seed=0):
    """Bundles of 64 rows as in ``bundle``; row i is linked to i - d and i + d for every distance d (64 among
    them, so that a bundle is a dependency level), one row in 64 reads ``hub`` earlier and as many later rows
    besides; columns in any order."""
    rng = np.random.default_rng(seed)
    col, row = [], [0]
    for i in range(n):
        c = {j for d in dists for j in (i - d, i + d) if 0 <= j < n}
        if hub and i % 64 == 7 and i > 64:
            c |= {int(j) for j in rng.integers(0, i - i % 64, hub)}
            c |= {int(j) for j in rng.integers(min(i - i % 64 + 64, n - 1), n, hub) if j > i}
        col += list(rng.permutation(sorted(c)))
        row.append(len(col))
    row = np.array(row, np.int32)
    off = rng.uniform(0.1, 1.0, len(col))
    diag = -1.1 * np.add.reduceat(off, row[:-1]) - 0.1
    return dict(n_self=n, n_total=n, row=row, col=np.array(col, np.int32), diag=diag, off=off,
                b=rng.uniform(-1, 1, n))


def ring_distances(m, back):
    """For every entry that reads a value updated in the same sweep: the rows of the schedule between that
    value and the end of the reader's dependency level, and the entry's place in its row."""
    n, row, col = m["n_self"], m["row"], m["col"]
    level = np.zeros(n, int)
    for i in range(n):   # (the backward sweep takes the forward schedule from its end)
        c = col[row[i]:row[i + 1]]
        level[i] = level[c[c < i]].max(initial=-1) + 1
    order = np.lexsort((np.arange(n), level))
    place = np.empty(n, int)
    place[order] = np.arange(n)
    if back:
        place, level = n - 1 - place, level.max() - level
    end = np.cumsum(np.bincount(level))
    i = np.repeat(np.arange(n), np.diff(row))
    new = col > i if back else col < i
    return (end[level[i]] - place[col])[new], (np.arange(len(col)) - row[i])[new]


NEAR = tuple(range(64, 640, 64))


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("dists,hub,longest", [((64, 4064, 8160), 0, 8), ((64, 128, 4064, 8160, 9600), 0, 8),
                                               (NEAR[:5] + (4064, 8160, 9600, 9664), 0, 16),
                                               (NEAR + (4064, 8160), 0, 24), ((64, 4064, 8160), 30, 70)])
def test_values_that_left_the_ring(dists, hub, longest, prec):
    """The ring in LDS holds the last 4,096 new values in FP64, 8,192 in FP32: links that reach just inside
    it, just past it and far past it, in rows of each shape of the kernel (8, 16 and 24 entries loaded
    ahead, and entries past those). Against the level-by-level launches: same bits."""
    m = layered(12800, dists, hub)
    ring = 8192 if prec else 4096
    assert longest - 8 < np.diff(m["row"]).max() <= longest
    for back in (False, True):
        dist, k = ring_distances(m, back)
        assert (dist > ring).sum() > 1000 and (dist <= ring).sum() > 1000
        assert {ring, ring + 1} <= set(dist)
        assert not hub or ((dist > ring) & (k >= 24)).sum() > 100
    res = []
    for flow in (0, 1):
        a = gpu_amg(gsOrdering=0, precision=prec, nMaxIterations=5, relativeTolerance=1e-30)
        a.set_tuning("exact_flow", flow)
        ls = ls_from(m)
        a.solve(ls)
        res.append((ls.delta.copy(), a.history()))
        assert a.get_tuning("exact_flow_wg_levels") & 1 == flow
    assert np.array_equal(res[0][0], res[1][0]) and np.array_equal(res[0][1], res[1][1])


@pytest.mark.parametrize("n", [2, 15, 16, 17, 33, 127, 255, 256])
def test_direct_level_inverse_at_panel_edges(n):
    """The blocked inverse of the direct level, at the edges of its panels and at its limit."""
    rng = np.random.default_rng(n)
    m = matgen.chain(2 * n)
    m["off"] = rng.uniform(0.2, 2.0, len(m["off"]))
    sums = np.add.reduceat(m["off"], m["row"][:-1])
    m["diag"] = -sums * rng.uniform(0.7, 1.5, 2 * n)          # not dominant everywhere: rows are pivoted
    a = gpu_amg(gsOrdering=1, precision=1)
    a.setup(ls_from(m))
    d = a.direct_level(with_inverse=True)
    assert d["level"] == 1 and d["n"] <= 256
    L = a.level(1)
    A = np.diag(L["diag"])
    for i in range(d["n"]):
        for p in range(L["row"][i], L["row"][i + 1]):
            A[i, L["col"][p]] += L["off"][p]
    ref = np.linalg.inv(A)
    # backward error of elimination: n eps cond, and the growth of a few
    bound = 20 * d["n"] * 2.3e-16 * np.linalg.cond(A)
    assert np.abs(d["inv"] - ref).max() <= bound * np.abs(ref).max()
