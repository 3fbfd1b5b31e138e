"""The span walk's hit record on a fresh context: a first join whose record
outgrows the space by several times reports the whole demand, so that the
next join of the same data replays; the replayed rows are the evaluated
ones, in the same order where the order is defined (full stencil)."""
import numpy as np
import pytest

import oracle as O
import sjamd
from sjamd import datasets as D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("schedule", [sjamd.STRIDED, sjamd.WORKQUEUE])
def test_second_join_replays_after_a_record_many_times_too_large(schedule):
    pts, eps = D.uniform(60_000, 4, 41), 0.24
    roff, rids = O.join(pts, 4, eps, O.LID, sort_rows=True)
    assert int(roff[-1]) > 4 * max(1 << 23, 16 * len(pts))  # one word per ordered pair
    print(f"[span record] |S|={int(roff[-1])}", flush=True)
    ctx = sjamd.Context(0)
    try:
        g = ctx.grid_build(pts, 4, eps)
        for rep in (0, 1):
            r = g.join(form="full", schedule=schedule, sort_rows=True)
            assert r.stats()["fill_from_record"] == rep
            off, ids = r.csr()
            r.free()
            np.testing.assert_array_equal(off, roff)
            np.testing.assert_array_equal(ids, rids)
        g.free()
    finally:
        ctx.close()


CASES = {"uniform_4d": (20_000, 4, 0.1), "uniform_6d": (20_000, 6, 0.28), "uniform_8d": (6_000, 8, 0.45)}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("prec", [sjamd.FP64, sjamd.FP32_RECHECK])
def test_replayed_rows_are_the_evaluated_rows(ctx, name, prec):
    n, k, eps = CASES[name]
    pts = D.uniform(n, k, 43)
    roff, rids = O.join(pts, k, eps, O.LID, sort_rows=True)
    g = ctx.grid_build(pts, k, eps)
    for form in ("full", "unicomp", "bunicomp", "lid"):
        for cap in (0, int(roff[-1]) // 4 + 1):
            got = []
            for rec in (True, True, False):
                r = g.join(form=form, precision=prec, hit_record=rec, capacity=cap)
                assert r.stats()["fill_from_record"] == int(rec), (form, cap)
                got.append(r.csr())
                r.free()
            for off, ids in got:
                np.testing.assert_array_equal(off, roff)
                if form == "full":  # a defined order without the row sort
                    np.testing.assert_array_equal(ids, got[0][1])
                off, ids = O.csr_rows_sorted(np.asarray(off, dtype=np.uint64), np.asarray(ids, dtype=np.int32))
                np.testing.assert_array_equal(ids, rids)
    g.free()
