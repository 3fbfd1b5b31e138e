"""Canonical row order (sort_rows) at the sizes where the row sort changes
its network: rows of 1 to 5001 IDs, against the rows known by construction
(groups of points at one place, far from each other)."""
import numpy as np
import pytest

import sjamd

pytestmark = pytest.mark.gpu

SIZES = {
    # four rows of <= 16, two of <= 32, one of <= 64 per wave, and mixes
    "short": list(range(1, 70)) + [16] * 40 + [17] * 9 + [32] * 33 + [33] * 5 + [64] * 7,
    # 2, 4, 8 and 16 IDs per lane
    "registers": [65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1024],
    # runs of 1024 merged in memory: remainders and whole powers of two
    "merged": [1025, 2047, 2048, 2049, 3000, 4096, 5001],
}


@pytest.mark.parametrize("form", ["full", "lid"])
@pytest.mark.parametrize("kind", list(SIZES))
def test_rows_sorted_at_network_edges(kind, form):
    rng = np.random.default_rng(11)
    sizes = SIZES[kind]
    label = np.repeat(np.arange(len(sizes)), sizes)
    pts = np.stack([label * 4.0, np.zeros(label.size)], 1) + rng.random((label.size, 2)) * 0.1
    perm = rng.permutation(label.size)
    pts, label = pts[perm], label[perm]
    ctx = sjamd.Context(0)
    try:
        r = ctx.self_join(pts, 2, 1.0, form=form, sort_rows=True)
        off, ids = r.csr()
        r.free()
    finally:
        ctx.close()
    rows = [np.flatnonzero(label == g) for g in range(len(sizes))]
    assert int(off[-1]) == sum(c * c for c in sizes)
    for p in range(label.size):
        assert np.array_equal(ids[int(off[p]):int(off[p + 1])], rows[label[p]]), (p, sizes[label[p]])
