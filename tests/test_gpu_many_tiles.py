"""67.9 million points, each in a cell row of its own: more than 2^26 tiles
and sampled points, so that one lane per neighbour row or stencil cell would
ask for more than 2^32 threads in a launch.  Every point's only neighbour is
itself."""
import numpy as np
import pytest

import sjamd

pytestmark = pytest.mark.gpu


def test_more_tiles_than_a_launch_has_waves():
    import torch

    side, k, eps = 408, 4, 1.0
    n = side ** 3
    i = torch.arange(n, device="cuda")
    x = torch.zeros(n, 5, dtype=torch.float64, device="cuda")
    for j in range(3):  # dims 1..3: 1.73 eps apart
        x[:, 1 + j] = (i // side ** j % side).double() * 1.73
    del i
    torch.cuda.synchronize()
    ctx = sjamd.Context(0)
    try:
        print(f"[many tiles] {n} points", flush=True)
        g = ctx.grid_build(x, k, eps)
        est = g.batch_estimate(stride=1)
        assert est["sample_count"] == n
        print("[many tiles] join", flush=True)
        r = g.join(form="lid")
        assert r.total == n
        off, ids, rows = r.device_table()
        ids = sjamd.download(ids, n, np.int32)
        assert np.array_equal(sjamd.download(off, n + 1, np.uint64), np.arange(n + 1, dtype=np.uint64))
        assert np.array_equal(sjamd.download(rows, n, np.uint32).astype(np.int32), ids)
        ids.sort()
        assert np.array_equal(ids, np.arange(n, dtype=np.int32))
        r.free()
        g.free()
    finally:
        ctx.close()
        del x
        torch.cuda.empty_cache()
