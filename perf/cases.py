"""Performance cases of the epsilon self-join: what users of the framework
have it do, through its Python and C entry points.

A case is one of five kinds of program:
  join    points on the device -> neighbour table on the device
          (Context.self_join, then the device table in cell order or the
          device CSR in point order);
  rounds  the reference program's flow: grid, batch estimate, join in result
          rounds of the estimated buffer size, neighbour table on the host;
  static  the allocation-free entry point into the caller's own arrays;
  many    one replay of a planned batch of independent joins.

Rows are asked for in canonical order (sort_rows) wherever a form mirrors
pairs, since such rows otherwise have no fixed order; the full stencil and
the many-join batch (which has no row sort) use the order that they produce,
which is the same on every run.  All outputs are whole numbers (offsets and
point IDs), so no case has values to compare with 64-bit arithmetic: they
are equal or wrong.  A pass ends with the neighbour IDs in the program's own
array, whose length does not depend on the number of pairs found (as a
program's later, fixed-shape steps need it).
"""
import ctypes
import json
import math
import os
import statistics
import sys
import weakref

import numpy
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "self-join-hpbdc2019_amd"))

import sjamd  # noqa: E402

LAMBDA = 40.0    # rate of the clipped exponential points
CLUSTERS = 100   # Gaussian clusters, centres in [0, 10]^d
SIGMA = 0.5
BOX = 10.0

JOIN = dict(kind="join", points="uniform", form="lid", schedule="strided", precision="fp64", view="table")


def _join(**kw):
    c = dict(JOIN, **kw)
    c.setdefault("k", c["d"])
    return c


def listed():
    return [
        # the smallest calls: a program that joins many small point sets one
        # after another, where launches and waits count
        _join(name="tiny_2d_1k", n=1_000, d=2, mean=8.0),
        # the small benchmark configuration (100,000 uniform points, about 9
        # neighbours each), its table read back in point order
        _join(name="uniform2d_100k", n=100_000, d=2, mean=7.9, form="unicomp", view="csr"),
        # the headline configuration: skewed 2-D points through the work
        # queue in the precision form, rows in canonical order
        _join(name="exp2d_2m", n=2_000_000, d=2, points="exp", mean=64.0, form="bunicomp", schedule="queue",
              precision="fp32"),
        # the reference's full-stencil work queue (its modes 7 and 9) on an
        # odd number of points, rows as produced
        _join(name="exp2d_full_1m", n=999_983, d=2, points="exp", mean=64.0, form="full", schedule="queue"),
        # an ordinary 3-D catalogue join in plain FP64, table in point order
        _join(name="exp3d_500k", n=524_287, d=3, points="exp", mean=48.0, view="csr"),
        # the 6-D benchmark configuration in the precision form
        _join(name="uniform6d_2m", n=2_000_000, d=6, mean=32.0, precision="fp32"),
        # the highest tiled dimension: few cells per dimension, most
        # candidates miss
        _join(name="uniform8d_100k", n=100_003, d=8, mean=24.0, schedule="queue"),
        # feature vectors: 64-D clusters indexed in 6 dimensions, on the
        # matrix cores
        _join(name="clusters64d_500k", n=500_000, d=64, k=6, points="clusters", mean=50.0, precision="fp32"),
        # feature vectors of odd width in plain FP64
        _join(name="clusters17d_60k", n=60_001, d=17, k=5, points="clusters", mean=50.0),
        # the reference program: estimate, result rounds, host neighbour table
        dict(name="rounds4d_300k", kind="rounds", n=300_000, d=4, k=4, points="uniform", mean=40.0, form="lid",
             schedule="strided", precision="fp64"),
        # a loop that may not allocate: the join into the caller's arrays
        dict(name="static2d_50k", kind="static", n=50_000, d=2, k=2, points="uniform", mean=24.0, form="lid",
             schedule="strided", precision="fp64"),
        # a planned batch of joins of mixed size, dimension and density
        dict(name="many12", kind="many", count=12, n_lo=10_000, n_hi=300_000, dims="2,3,4,6,8", mean_lo=8.0,
             mean_hi=64.0, form="full", schedule="queue", precision="fp32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above."""
    kind = rng.choice(["join"] * 6 + ["wide"] * 2 + ["rounds", "static", "many"])
    prec = rng.choice(["fp64", "fp32"])
    sched = rng.choice(["strided", "queue"])
    form = rng.choice(["full", "unicomp", "bunicomp", "lid"])
    if kind == "join":
        d = rng.choice([2, 2, 3, 4, 6, 8])
        top = {2: 2_000_000, 3: 2_000_000, 4: 1_000_000, 6: 1_000_000, 8: 150_000}[d]
        return _join(n=_log_int(rng, 1_000, top), d=d, points=rng.choice(["uniform", "exp"]),
                     mean=round(rng.uniform(8.0, 64.0), 2), form=form, schedule=sched, precision=prec,
                     view=rng.choice(["table", "csr"]))
    if kind == "wide":
        d = rng.randint(9, 64)
        n = _log_int(rng, 10_000, 400_000 if prec == "fp32" else 60_000)
        return _join(n=n, d=d, k=rng.randint(4, 6), points="clusters", mean=round(rng.uniform(8.0, 64.0), 2),
                     form=rng.choice(["full", "lid"]), schedule=sched, precision=prec,
                     view=rng.choice(["table", "csr"]))
    if kind == "rounds":
        d = rng.choice([2, 3, 4])
        return dict(kind="rounds", n=_log_int(rng, 20_000, 400_000), d=d, k=d,
                    points=rng.choice(["uniform", "exp"]), mean=round(rng.uniform(8.0, 48.0), 2), form=form,
                    schedule=sched, precision=prec)
    if kind == "static":
        d = rng.choice([2, 3])
        return dict(kind="static", n=_log_int(rng, 1_000, 500_000), d=d, k=d,
                    points=rng.choice(["uniform", "exp"]), mean=round(rng.uniform(8.0, 48.0), 2), form=form,
                    schedule=sched, precision=prec)
    return dict(kind="many", count=rng.randint(4, 16), n_lo=10_000, n_hi=_log_int(rng, 50_000, 250_000),
                dims=rng.choice(["2,3,4,6,8", "2,3", "2,3,4,6"]), mean_lo=8.0,
                mean_hi=round(rng.uniform(32.0, 64.0), 2), form="full", schedule=sched, precision=prec)


# ------------------------------------------------------------------ inputs
def _eps(points, n, d, mean):
    """eps for about `mean` neighbours per point (the point included)."""
    if points == "clusters":
        # same-cluster distances: d2 = 2 sigma^2 chi2_d (Wilson-Hilferty
        # quantile of the share of the cluster that is to be within eps)
        p = min(0.5, mean / (n / CLUSTERS))
        z = statistics.NormalDist().inv_cdf(p)
        c = 2.0 / (9.0 * d)
        return SIGMA * math.sqrt(2.0 * d * max(0.01, 1.0 - c + z * math.sqrt(c)) ** 3)
    ball = math.pi ** (d / 2) / math.gamma(d / 2 + 1)
    density = (LAMBDA / 2) ** d if points == "exp" else 1.0  # mean density at a point
    return (mean / (n * ball * density)) ** (1.0 / d)


def _points(points, n, d, gen):
    if points == "clusters":
        centres = BOX * torch.rand(CLUSTERS, d, generator=gen, dtype=torch.float64, device="cuda")
        label = torch.randint(CLUSTERS, (n,), generator=gen, device="cuda")
        return centres[label] + SIGMA * torch.randn(n, d, generator=gen, dtype=torch.float64, device="cuda")
    u = torch.rand(n, d, generator=gen, dtype=torch.float64, device="cuda")
    return torch.clamp(-torch.log1p(-u) / LAMBDA, max=1.0) if points == "exp" else u


def _instances(case):
    """(n, d, points, mean) of each join of a many-join case."""
    dims = [int(v) for v in case["dims"].split(",")]
    m = case["count"]
    out = []
    for i in range(m):
        t = i / max(1, m - 1)
        d = dims[i % len(dims)]
        n = int(round(case["n_lo"] * (case["n_hi"] / case["n_lo"]) ** t))
        n = min(n, 100_000) if d == 8 else n
        mean = case["mean_lo"] + (case["mean_hi"] - case["mean_lo"]) * ((i * 5) % m) / m
        out.append((n, d, "exp" if i % 2 else "uniform", mean))
    return out


# one context for the states of one case, as a program keeps one: it lives
# while any of them does
_contexts = weakref.WeakValueDictionary()


def _context(case):
    key = json.dumps({k: v for k, v in case.items() if k != "name"}, sort_keys=True)
    ctx = _contexts.get(key)
    if ctx is None:
        ctx = _contexts[key] = sjamd.Context(torch.cuda.current_device())
    return ctx


def _options(case):
    return dict(form=case["form"], precision=sjamd.FP32_RECHECK if case["precision"] == "fp32" else sjamd.FP64,
                schedule=sjamd.WORKQUEUE if case["schedule"] == "queue" else sjamd.STRIDED)


def _capacity(pairs):
    """Length of the array in which a program keeps about `pairs` IDs."""
    return int(1.5 * pairs) + 65_536


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ctx = _context(case)
    kw = _options(case)
    st = dict(case=case, ctx=ctx, last=None)
    if case["kind"] == "many":
        shapes = _instances(case)
        sets = [(_points(p, n, d, gen), d, _eps(p, n, d, mean)) for n, d, p, mean in shapes]
        torch.cuda.synchronize()
        st["plan"] = ctx.many(sets, **kw)
        st["ids"] = torch.zeros(_capacity(sum(n * mean for n, _, _, mean in shapes)), dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        return st
    n, d = case["n"], case["d"]
    st["x"] = _points(case["points"], n, d, gen)
    st["eps"] = _eps(case["points"], n, d, case["mean"])
    st["kw"] = dict(kw, sort_rows=case["form"] != "full")
    cap = _capacity(n * case["mean"])
    if case["kind"] == "rounds":
        st["ids"] = numpy.zeros(cap, dtype=numpy.int32)
    else:
        st["ids"] = torch.zeros(cap, dtype=torch.int32, device="cuda")
    if case["kind"] == "static":
        st["params"] = sjamd.make_params(**st["kw"])
        st["offsets"] = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
        st["rows"] = torch.zeros(n, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    return st


# ------------------------------------------------------------------ passes
class _View:
    """A device array of the library as torch sees it, without a copy.  The
    tensor made of it keeps the view, and the view the owner of the memory
    (the result or plan, and through it the context)."""

    def __init__(self, owner, ptr, count, kind):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(count,), typestr=kind, data=(ptr, False), version=2, strides=None)


def _tensor(owner, ptr, count, kind):
    return torch.as_tensor(_View(owner, ptr, count, kind), device="cuda")


def _keep(st, ids):
    """The neighbour IDs into the program's own array of fixed length."""
    st["ids"][:ids.numel()].copy_(ids)
    return st["ids"]


def _run_join(st):
    case = st["case"]
    if st["last"] is not None:
        st["last"].free()  # the previous pass's table
    r = st["last"] = st["ctx"].self_join(st["x"], case["k"], st["eps"], **st["kw"])
    if case["view"] == "csr":
        off, ids = r.device_csr()
        return _tensor(r, off, r.n + 1, "<i8"), _keep(st, _tensor(r, ids, r.total, "<i4"))
    off, ids, rows = r.device_table()
    return (_tensor(r, off, r.n + 1, "<i8"), _keep(st, _tensor(r, ids, r.total, "<i4")),
            _tensor(r, rows, r.n, "<i4"))


def _run_rounds(st):
    # rounds of any form are asked for in canonical order
    g = st["ctx"].grid_build(st["x"], st["case"]["k"], st["eps"])
    est = g.batch_estimate()
    r = g.join(**dict(st["kw"], sort_rows=True, capacity=est["buffer_size"]))
    table = r.neighbor_table()
    # the rounds' neighbour IDs one after another in the program's array
    ptr, cnt, at = ctypes.c_void_p(), ctypes.c_uint64(), 0
    for b in range(int(table[:, 3].max()) + 1):
        rc = sjamd.lib().sj_result_batch_data(r.h, b, ctypes.byref(ptr), ctypes.byref(cnt))
        if rc != 0:
            raise sjamd.SJError(rc, sjamd.lib().sj_last_error().decode())
        st["ids"][at:at + cnt.value] = numpy.frombuffer((ctypes.c_int32 * cnt.value).from_address(ptr.value),
                                                        dtype=numpy.int32)
        at += cnt.value
    r.free()
    g.free()
    return dict(table=table, ids=st["ids"])


def _run_static(st):
    case, x = st["case"], st["x"]
    total = ctypes.c_uint64()
    rc = sjamd.lib().sj_self_join_static(
        st["ctx"].h, ctypes.c_void_p(x.data_ptr()), case["n"], case["d"], case["k"], float(st["eps"]),
        ctypes.byref(st["params"]), ctypes.c_void_p(st["offsets"].data_ptr()), ctypes.c_void_p(st["ids"].data_ptr()),
        st["ids"].numel(), ctypes.c_void_p(st["rows"].data_ptr()), ctypes.byref(total))
    if rc != 0:
        raise sjamd.SJError(rc, sjamd.lib().sj_last_error().decode())
    return st["offsets"], st["ids"], st["rows"]


def _run_many(st):
    plan = st["plan"]
    plan.run()
    out, at = [], 0
    for i in range(len(plan)):
        off, ids, rows, total = plan.device_table(i)
        n = plan.shapes[i][0]
        st["ids"][at:at + total].copy_(_tensor(plan, ids, total, "<i4"))
        at += total
        out.append((_tensor(plan, off, n + 1, "<i8"), _tensor(plan, rows, n, "<i4")))
    return dict(ids=st["ids"], tables=out)


_RUN = dict(join=_run_join, rounds=_run_rounds, static=_run_static, many=_run_many)


def run(st):
    return _RUN[st["case"]["kind"]](st)


def work(case):
    """Coordinates read once, offsets, row IDs and neighbour IDs written
    once; the distance of every unordered result pair (3d - 1 operations)."""
    if case["kind"] == "many":
        sets = [(n, d, mean) for n, d, _, mean in _instances(case)]
    else:
        sets = [(case["n"], case["d"], case["mean"])]
    return dict(bytes=sum(n * d * 8 + (n + 1) * 8 + n * 4 + n * mean * 4 for n, d, mean in sets),
                flops=sum(n * mean / 2 * (3 * d - 1) for n, d, mean in sets))
