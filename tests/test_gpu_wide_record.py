"""The wide FP64 walk's fill replayed from the count's hit record: whole
results and result rounds equal the oracle's, at the edges of its
32-candidate chunks and 64-point tiles."""
import numpy as np
import pytest

import oracle as O
import sjamd
from sjamd import datasets as D

pytestmark = pytest.mark.gpu

CASES = {
    "d9_k9_33": lambda: (D.uniform(33, 9, 1), 4, 0.9),
    "d17_k5_4k": lambda: (D.clusters(4001, 17, 2), 5, 2.6),
    "d64_k3_2k": lambda: (D.clusters(2000, 64, 3), 3, 5.2),
    "d5_k2_same": lambda: (np.full((200, 5), 1.5), 2, 0.5),
    "d6_k4_3k": lambda: (D.uniform(3000, 6, 4), 4, 0.25),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("form", ["full", "unicomp", "bunicomp", "lid"])
def test_wide_replay_matches_oracle(name, form):
    pts, k, eps = CASES[name]()
    roff, rids = O.join(pts, k, eps, O.LID, sort_rows=True)
    ctx = sjamd.Context(0)
    try:
        g = ctx.grid_build(pts, k, eps)
        for kw in (dict(), dict(), dict(schedule=sjamd.WORKQUEUE), dict(hit_record=False),
                   dict(capacity=max(int(roff[-1]) // 3, int(np.diff(roff.astype(np.int64)).max())) + 1)):
            r = g.join(form=form, sort_rows=True, **kw)
            assert r.stats()["fill_from_record"] == (0 if "hit_record" in kw else 1), kw
            off, ids = r.csr()
            r.free()
            np.testing.assert_array_equal(off, roff, err_msg=str(kw))
            np.testing.assert_array_equal(ids, rids, err_msg=str(kw))
        g.free()
    finally:
        ctx.close()
