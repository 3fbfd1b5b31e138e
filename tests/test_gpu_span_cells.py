"""The span walk where squared distances of different points underflow to 0
(eps below 1e-162): only points of adjacent cells are neighbours, however
many cells apart the canonical distance is 0.  Lattices with spacing eps, 8
and 5 cells wide, single joins and a batch, against the oracle."""
import itertools

import numpy as np
import pytest

import oracle as O
import sjamd

pytestmark = pytest.mark.gpu


def _lattice(side, k, eps):
    return np.array(list(itertools.product(range(side), repeat=k)), dtype=np.float64) * eps


CASES = {"8x4d_1e-170": (8, 4, 1e-170), "5x5d_1e-165": (5, 5, 1e-165), "8x4d_1e-163": (8, 4, 1e-163)}


@pytest.mark.parametrize("name", list(CASES))
def test_underflowing_distances(ctx, name):
    side, k, eps = CASES[name]
    pts = _lattice(side, k, eps)
    roff, rids = O.join(pts, k, eps, O.LID, sort_rows=True)
    print(f"[span cells] {name} |S|={int(roff[-1])}", flush=True)
    assert O.eps_threshold(eps) == 0.0
    g = ctx.grid_build(pts, k, eps)
    for form in ("full", "unicomp", "bunicomp", "lid"):
        for prec in (sjamd.FP64, sjamd.FP32_RECHECK):
            for kw in (dict(), dict(hit_record=False), dict(capacity=int(roff[-1]) // 3 + 1000)):
                r = g.join(form=form, precision=prec, sort_rows=True, **kw)
                off, ids = r.csr()
                r.free()
                tag = f"{name} {form} prec={prec} {kw}"
                np.testing.assert_array_equal(off, roff, err_msg=tag)
                np.testing.assert_array_equal(ids, rids, err_msg=tag)
    g.free()


@pytest.mark.parametrize("prec", [sjamd.FP64, sjamd.FP32_RECHECK])
def test_underflowing_distances_in_a_batch(ctx, prec):
    sets = [(_lattice(s, k, e), k, e) for s, k, e in CASES.values()]
    m = ctx.many(sets, form="lid", precision=prec)
    for i, (pts, k, eps) in enumerate(sets):
        roff, rids = O.join(pts, k, eps, O.LID, sort_rows=True)
        off, ids = m.csr(i)
        off, ids = O.csr_rows_sorted(np.asarray(off, dtype=np.uint64), np.asarray(ids, dtype=np.int32))
        np.testing.assert_array_equal(off, roff, err_msg=str(i))
        np.testing.assert_array_equal(ids, rids, err_msg=str(i))
    m.free()
