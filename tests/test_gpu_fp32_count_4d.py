"""sj_stats.fp32_misclassified of the span walk against a host count.

4-D points on the 2^-10 lattice (coordinates below 2^24 units), so that every
difference and every coordinate minus a tile centre is exact in FP32: the
plain FP32 squared distance (FMA chain of the differences, dimension order)
depends on the pair alone and the host reproduces it.  Pairs lie at integer
offsets whose squared length is within 8 of 2^26 lattice units (eps = 8), where
FP32 rounds many of them across the threshold; the groups are 24 eps apart.
The full stencil meets every ordered pair once."""
import numpy as np
import pytest

import oracle as O
import sjamd
from fp32emu import F32, fma32

pytestmark = pytest.mark.gpu

EPS, UNIT = 8.0, 2.0 ** -10


def _points():
    rng = np.random.default_rng(3)
    target, vecs = 1 << 26, []
    while len(vecs) < 400:
        v = rng.integers(1000, 4700, 3)
        rest = target - int((v * v).sum())
        w = int(round(np.sqrt(rest)))
        if abs(w * w - rest) <= 8:
            vecs.append(v.tolist() + [w])
    pts = []
    for g, v in enumerate(vecs):
        at = np.array([g % 5, g // 5 % 5, g // 25 % 4, g // 100]) * 24 * 8 * 1024
        pts += [at, at + v]
    return np.array(pts, dtype=np.float64) * UNIT


def _host_count(pts):
    T = O.eps_threshold(EPS)
    p, q = pts[0::2], pts[1::2]
    f = (q - p).astype(F32)  # exact
    s32 = (f[:, 0] * f[:, 0]).astype(F32)
    for j in range(1, 4):
        s32 = fma32(f[:, j], f[:, j], s32)
    return 2 * int(((s32 <= F32(T)) != (O.dist2_batch(p, q) <= T)).sum())


def test_fp32_misclassified_of_the_span_walk(ctx):
    pts = _points()
    want = _host_count(pts)
    print(f"[fp32 count 4-D] {len(pts)} points, {want} wrong FP32 decisions", flush=True)
    assert want > 20
    roff, rids = O.join(pts, 4, EPS, O.LID, sort_rows=True)
    for form, share in (("full", 1), ("lid", 2)):
        r = ctx.self_join(pts, 4, EPS, form=form, precision=sjamd.FP32_RECHECK, sort_rows=True)
        st = r.stats()
        off, ids = r.csr()
        r.free()
        np.testing.assert_array_equal(off, roff)
        np.testing.assert_array_equal(ids, rids)
        # LID meets a pair of different cells once, one of a cell twice
        assert want // share <= st["fp32_misclassified"] <= want
        if share == 1:
            assert st["fp32_misclassified"] == want
        assert st["fp32_band_pairs"] >= want // share
    m = ctx.many([(pts, 4, EPS)], form="full", precision=sjamd.FP32_RECHECK)
    assert m.stats()["fp32_misclassified"] == want
    m.free()
