"""The allocation-free entry point in 4-D at sizes where its scratch is
nearly used up: the grid's dense lookup table grows step by step until it no
longer fits beside the join's share, and no step may leave the join short."""
import ctypes as C

import numpy as np
import pytest

import sjamd

pytestmark = pytest.mark.gpu


# (points, schedule, lengths of the box in dim 0): 57^3 cells per unit of
# length, 0.7 MiB of table per step
CASES = [(1_000_000, sjamd.STRIDED, 240), (1_000_000, sjamd.WORKQUEUE, 240), (1_300_000, sjamd.STRIDED, 180)]


@pytest.mark.parametrize("n,schedule,longest", CASES)
def test_dense_table_leaves_room_for_the_join(ctx, n, schedule, longest):
    import torch

    L = sjamd.lib()
    params = sjamd.make_params(form="lid", schedule=schedule, sort_rows=True)
    need = L.sj_static_need(n, 4, 4, C.byref(params))
    assert need <= L.sj_static_scratch_bytes()  # accepted by the entry point's size check
    print(f"[static 4-D] n={n} schedule={schedule} need={need}", flush=True)
    u = torch.rand(n, 4, generator=torch.Generator(device="cuda").manual_seed(n), dtype=torch.float64, device="cuda")
    cap = 8 * n  # about 5 neighbours per point in the shortest box
    off = torch.empty(n + 1, dtype=torch.int64, device="cuda")
    ids = torch.empty(cap, dtype=torch.int32, device="cuda")
    rows = torch.empty(n, dtype=torch.int32, device="cuda")
    tot = C.c_uint64()
    for length in range(12, longest):
        x = u * torch.tensor([float(length), 54.0, 54.0, 54.0], dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        rc = L.sj_self_join_static(ctx.h, C.c_void_p(x.data_ptr()), n, 4, 4, 1.0, C.byref(params),
                                   C.c_void_p(off.data_ptr()), C.c_void_p(ids.data_ptr()), cap,
                                   C.c_void_p(rows.data_ptr()), C.byref(tot))
        assert rc == 0, (length, L.sj_last_error())
        if length % 24 and length + 1 < longest:
            continue
        r = ctx.self_join(x, 4, 1.0, form="lid", schedule=schedule, sort_rows=True)
        o, i, rid = r.device_table()
        assert tot.value == r.total
        np.testing.assert_array_equal(off.cpu().numpy().astype(np.uint64), sjamd.download(o, n + 1, np.uint64))
        np.testing.assert_array_equal(ids[:r.total].cpu().numpy(), sjamd.download(i, r.total, np.int32))
        np.testing.assert_array_equal(rows.cpu().numpy().astype(np.uint32), sjamd.download(rid, n, np.uint32))
        r.free()
