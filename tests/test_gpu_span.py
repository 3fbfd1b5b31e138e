"""The span walk (d = k >= 4) against the oracle where its tiles, blocks and
buffers have edges: fewer points than a block of 16, tiles of 63 to 65
points, points at one place (every pair passes, rows above the pair buffer),
pairs at exactly eps, sparse grids, and coordinates beyond the matrix-core
filter's range.  Every form, both precisions, replayed and evaluated fills."""
import itertools

import numpy as np
import pytest

import oracle as O
import sjamd
from sjamd import datasets as D

pytestmark = pytest.mark.gpu


def _lattice(side, k):
    return np.array(list(itertools.product(range(side), repeat=k)), dtype=np.float64)


CASES = {
    "one_point_4d": lambda: (D.uniform(1, 4, 1), 0.5),
    "seven_points_8d": lambda: (D.uniform(7, 8, 2), 0.9),
    "tile_63_5d": lambda: (D.uniform(63, 5, 3), 2.0),
    "tile_64_6d": lambda: (D.uniform(64, 6, 4), 2.0),
    "tile_65_7d": lambda: (D.uniform(65, 7, 5), 2.0),
    "one_place_1500_4d": lambda: (np.full((1500, 4), 0.25), 0.1),
    "lattice_eps1_4d": lambda: (_lattice(6, 4), 1.0),
    "lattice_eps_sqrt2_5d": lambda: (_lattice(4, 5), float(np.sqrt(2.0))),
    "sparse_exp_6d": lambda: (D.exponential_clipped(6000, 6, 6), 0.01),
    "offset_1e6_4d": lambda: (D.uniform(5000, 4, 7) + 1e6, 0.12),
    "wide_1e16_4d": lambda: (D.uniform(3000, 4, 8) * 1e16, 1.5e15),
    "huge_1e150_5d": lambda: (D.uniform(2000, 5, 9) * 1e150, 2.5e149),
    "tiny_1e-20_4d": lambda: (D.uniform(3000, 4, 10) * 1e-20, 1.5e-21),
    "uniform_9k_7d": lambda: (D.uniform(9001, 7, 11), 0.31),
}


@pytest.mark.parametrize("name", list(CASES))
def test_span_walk_matches_oracle(ctx, name):
    pts, eps = CASES[name]()
    k = pts.shape[1]
    roff, rids = O.join(pts, k, eps, O.LID, sort_rows=True)
    print(f"[span] {name} n={pts.shape[0]} |S|={int(roff[-1])}", flush=True)
    g = ctx.grid_build(pts, k, eps)
    for form in ("full", "unicomp", "bunicomp", "lid"):
        for prec in (sjamd.FP64, sjamd.FP32_RECHECK):
            for kw in (dict(), dict(hit_record=False), dict(schedule=sjamd.WORKQUEUE)):
                r = g.join(form=form, precision=prec, sort_rows=True, **kw)
                off, ids = r.csr()
                r.free()
                tag = f"{name} {form} prec={prec} {kw}"
                np.testing.assert_array_equal(off, roff, err_msg=tag)
                np.testing.assert_array_equal(ids, rids, err_msg=tag)
    g.free()


@pytest.mark.parametrize("form", ["full", "bunicomp", "lid"])
def test_span_walk_in_rounds(ctx, form):
    """result rounds (windows of rows) from the record and evaluated again"""
    pts, eps = CASES["uniform_9k_7d"]()
    roff, rids = O.join(pts, 7, eps, O.LID, sort_rows=True)
    g = ctx.grid_build(pts, 7, eps)
    for kw in (dict(), dict(hit_record=False)):
        r = g.join(form=form, sort_rows=True, capacity=int(roff[-1]) // 5 + 1, **kw)
        assert r.stats()["num_batches"] >= 4
        off, ids = r.csr()
        r.free()
        np.testing.assert_array_equal(off, roff)
        np.testing.assert_array_equal(ids, rids)
    g.free()
