"""The span walk on cells with many points, where blocks of 16 candidates are
decided whole and recorded as masks: points in one cell, groups over several
cells with sparse points between (masks and single hits in one tile), whole
and partial blocks and tiles.  Every form, both precisions, replayed and
evaluated fills, result rounds and the order of full-stencil rows, against
the oracle."""
import numpy as np
import pytest

import oracle as O
import sjamd
from sjamd import datasets as D

pytestmark = pytest.mark.gpu


def _groups(sizes, k, spread, seed):
    """groups 3 apart in dim 0 and 1, points within spread of their corner"""
    rng = np.random.default_rng(seed)
    g = np.repeat(np.arange(len(sizes)), sizes)
    pts = spread * rng.random((g.size, k))
    pts[:, 0] += 3.0 * (g % 3)
    pts[:, 1] += 3.0 * (g // 3)
    return pts[rng.permutation(g.size)]


CASES = {
    "one_cell_4d": lambda: (_groups([1777], 4, 0.2, 1), 1.0),
    "one_cell_8d": lambda: (_groups([1031], 8, 0.3, 2), 1.0),
    "groups_4d": lambda: (_groups([65, 640, 129, 1000, 300], 4, 1.3, 3), 1.0),
    "groups_5d": lambda: (_groups([500, 17, 900], 5, 1.1, 4), 0.9),
    "groups_6d": lambda: (_groups([700, 64, 333], 6, 0.9, 5), 1.0),
    "groups_7d": lambda: (_groups([401, 402, 403], 7, 0.8, 6), 1.0),
    "uniform_4d": lambda: (D.uniform(3001, 4, 7), 0.45),
    "uniform_6d": lambda: (D.uniform(2001, 6, 8), 0.6),
}


@pytest.mark.parametrize("name", list(CASES))
def test_dense_cells_match_oracle(ctx, name):
    pts, eps = CASES[name]()
    k = pts.shape[1]
    roff, rids = O.join(pts, k, eps, O.LID, sort_rows=True)
    total, longest = int(roff[-1]), int(np.diff(roff.astype(np.int64)).max())
    g = ctx.grid_build(pts, k, eps)
    print(f"[span dense] {name} n={len(pts)} |S|={total}", flush=True)
    for form in ("full", "unicomp", "bunicomp", "lid"):
        rows = None
        for prec in (sjamd.FP64, sjamd.FP32_RECHECK):
            for kw in (dict(), dict(hit_record=False), dict(schedule=sjamd.WORKQUEUE),
                       dict(capacity=max(total // 5, longest) + 1),
                       dict(capacity=max(total // 5, longest) + 1, hit_record=False)):
                tag = f"{name} {form} prec={prec} {kw}"
                r = g.join(form=form, precision=prec, **kw)
                st = r.stats()
                off, ids = r.csr()
                r.free()
                assert st["fill_from_record"] == int("hit_record" not in kw), tag
                assert st["fp32_misclassified"] <= st["fp32_band_pairs"]
                np.testing.assert_array_equal(off, roff, err_msg=tag)
                if form == "full":  # a defined order without the row sort
                    rows = ids if rows is None else rows
                    np.testing.assert_array_equal(ids, rows, err_msg=tag)
                off, ids = O.csr_rows_sorted(np.asarray(off, dtype=np.uint64), np.asarray(ids, dtype=np.int32))
                np.testing.assert_array_equal(ids, rids, err_msg=tag)
    g.free()


def test_some_case_is_dense_enough():
    """the walk takes blocks whole from 64 points per occupied cell on"""
    dense = 0
    for make in CASES.values():
        pts, eps = make()
        cells = np.unique(((pts - (pts.min(0) - eps)) / eps).astype(np.int64), axis=0)
        dense += len(pts) >= 64 * len(cells)
    assert dense >= 4


@pytest.mark.parametrize("form", ["full", "lid"])
def test_dense_cells_in_a_batch(ctx, form):
    sets = [CASES[n]() for n in ("one_cell_4d", "groups_6d", "one_cell_8d")]
    m = ctx.many([(p, p.shape[1], e) for p, e in sets], form=form, precision=sjamd.FP32_RECHECK)
    for rep in range(2):
        for i, (pts, eps) in enumerate(sets):
            roff, rids = O.join(pts, pts.shape[1], eps, O.LID, sort_rows=True)
            off, ids = m.csr(i)
            off, ids = O.csr_rows_sorted(np.asarray(off, dtype=np.uint64), np.asarray(ids, dtype=np.int32))
            np.testing.assert_array_equal(off, roff)
            np.testing.assert_array_equal(ids, rids)
        m.run()
    m.free()
