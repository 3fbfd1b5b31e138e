"""Host checks of the filter of the walk for d = k = 4..8 (no GPU).

The walk hands a pair to the FP64 predicate only if it passes a norm
expansion in FP64 or FP32, so the filter must pass every pair that the
predicate accepts.  The tests emulate the kernel's arithmetic (centring,
norms, products in three summation orders, scaled norms, threshold) on pairs
within a few ulps of eps, near and far from the tile's first point, and on
pairs clearly outside, most of which it must reject."""
import numpy as np
import pytest

import oracle as O
import sjamd
from fp32emu import fma32


def _pairs(rng, m, d, eps, spread):
    """pairs within a few ulps of eps, the tile's first point within spread"""
    dirs = rng.normal(size=(m, d))
    dirs /= np.linalg.norm(dirs, axis=1, keepdims=True)
    p = rng.uniform(-spread, spread, size=(m, d))
    return p, p + dirs * (eps * (1.0 + rng.uniform(-4e-15, 4e-15, size=(m, 1))))


def _fma(a, b, c):
    return fma32(a, b, c) if a.dtype == np.float32 else a * b + c  # FP64: one rounding more than the kernel's


def _norm(V):
    """one partial sum per dim modulo 4, then the sum of the four"""
    part = []
    for l in range(4):
        nn = np.zeros(V.shape[0], dtype=V.dtype)
        for j in range(l, V.shape[1], 4):
            nn = _fma(V[:, j], V[:, j], nn)
        part.append(nn)
    return (part[0] + part[1]) + (part[2] + part[3])


def _accumulated(A, B, C):
    """C + A.B per row: forward, backward, and the products' sum added last"""
    out = []
    for order in (range(A.shape[1]), reversed(range(A.shape[1]))):
        acc = C.copy()
        for j in order:
            acc = _fma(A[:, j], B[:, j], acc)
        out.append(acc)
    dot = np.zeros_like(C)
    for j in range(A.shape[1]):
        dot = dot + A[:, j] * B[:, j]
    out.append(C + dot)
    return out


def _passes(p, q, centre, d, T, prec):
    t = np.float32 if prec == sjamd.FP32_RECHECK else np.float64
    R = 4.0 * max(np.abs(p).max(), np.abs(q).max()) + 2.0 * np.sqrt(T)
    usable, scale, T1 = sjamd.span_band(T, R, d, prec)
    assert usable and t(scale) == scale and t(T1) == T1 and T < T1 and 0.9 < scale < 1.0
    A, B = (p - centre).astype(t), (q - centre).astype(t)
    C = _norm(A) * t(scale)
    thr = t(T1) - _norm(B) * t(scale)
    return [acc <= thr for acc in _accumulated(t(-2) * A, B, C)]


CASES = [(d, eps, mult) for d in (4, 5, 6, 7, 8) for eps, mult in ((0.02, 1.0), (0.125, 6.0), (3.7, 64.0), (1e-9, 3.0))]


@pytest.mark.parametrize("prec", [sjamd.FP64, sjamd.FP32_RECHECK])
@pytest.mark.parametrize("d,eps,mult", CASES)
def test_filter_passes_every_accepted_pair(d, eps, mult, prec):
    rng = np.random.default_rng(3000 + d)
    T = O.eps_threshold(eps)
    p, q = _pairs(rng, 100_000, d, eps, mult * eps)
    centre = rng.uniform(-mult * eps, mult * eps, size=d)
    hit = O.dist2_batch(p, q) <= T
    assert hit.any() and (~hit).any()
    for ok in _passes(p, q, centre, d, T, prec):
        assert ok[hit].all()
    # pairs a little outside are rejected while the tile spans a few eps
    if mult <= 6.0:
        far = p + (q - p) * 1.01
        for ok in _passes(p, far, centre, d, T, prec):
            assert not ok.any()


@pytest.mark.parametrize("d,eps,mult", CASES)
def test_filter_passes_what_plain_fp32_accepts(d, eps, mult):
    """pairs around the FP32 threshold whose FP32 sum of squared differences
    accepts them, right or wrong (sj_stats.fp32_misclassified)"""
    rng = np.random.default_rng(4000 + d)
    T = O.eps_threshold(eps)
    centre = rng.uniform(-mult * eps, mult * eps, size=d)
    dirs = rng.normal(size=(200_000, d))
    dirs /= np.linalg.norm(dirs, axis=1, keepdims=True)
    p = rng.uniform(-mult * eps, mult * eps, size=dirs.shape)
    q = p + dirs * (eps * (1.0 + rng.uniform(-1e-6, 8e-6 * mult, size=(len(dirs), 1))))
    f = (q - centre).astype(np.float32) - (p - centre).astype(np.float32)
    s32 = f[:, 0] * f[:, 0]
    for j in range(1, d):
        s32 = fma32(f[:, j], f[:, j], s32)
    accepted = s32 <= np.float32(T)
    assert (accepted & (O.dist2_batch(p, q) > T)).any()
    for ok in _passes(p, q, centre, d, T, sjamd.FP32_RECHECK):
        assert ok[accepted].all()


@pytest.mark.parametrize("d,eps,mult", CASES)
def test_plain_fp32_errs_only_near_eps(d, eps, mult):
    """the count of wrong plain FP32 decisions looks only at pairs whose d2 is
    within u ((2.03 d + 8.02) (3 nq + 2 d2) + T) of T, u = 1.1 * 2^-24, nq the
    query's scaled norm"""
    rng = np.random.default_rng(5000 + d)
    T = O.eps_threshold(eps)
    centre = rng.uniform(-mult * eps, mult * eps, size=d)
    dirs = rng.normal(size=(200_000, d))
    dirs /= np.linalg.norm(dirs, axis=1, keepdims=True)
    p = rng.uniform(-mult * eps, mult * eps, size=dirs.shape)
    q = p + dirs * (eps * (1.0 + rng.uniform(-4e-6, 4e-6, size=(len(dirs), 1)) * mult))
    A, B = (p - centre).astype(np.float32), (q - centre).astype(np.float32)
    f = B - A
    s32 = f[:, 0] * f[:, 0]
    for j in range(1, d):
        s32 = fma32(f[:, j], f[:, j], s32)
    d2 = O.dist2_batch(p, q)
    wrong = (s32 <= np.float32(T)) != (d2 <= T)
    assert wrong.any()
    _, scale, _ = sjamd.span_band(T, 4.0 * mult * eps + 2.0 * eps, d, sjamd.FP32_RECHECK)
    nq = (_norm(A) * np.float32(scale)).astype(np.float64)
    near = np.abs(d2 - T) <= 1.1 * 2.0 ** -24 * ((2.03 * d + 8.02) * (3.0 * nq + 2.0 * d2) + T)
    assert near[wrong].all()


@pytest.mark.parametrize("prec", [sjamd.FP64, sjamd.FP32_RECHECK])
def test_filter_range(prec):
    """outside its range every pair goes to the predicate; inside it the
    threshold is finite in the filter's precision"""
    t = np.float32 if prec == sjamd.FP32_RECHECK else np.float64
    for eps in 10.0 ** np.arange(-170.0, 165.0, 2.5):
        T = O.eps_threshold(eps)
        for box in (0.0, 1.0, 1e10, 1e20, 1e160):
            R = box + 2.0 * eps  # a grid extends eps beyond the points on both sides
            usable, scale, T1 = sjamd.span_band(T, R, 6, prec)
            if usable:
                with np.errstate(over="ignore"):
                    assert np.isfinite(t(T1)) and np.isfinite(t(64.0) * t(R) * t(R))
                assert t(T) > 0
    assert not sjamd.span_band(0.0, 1.0, 4, prec)[0]
    assert not sjamd.span_band(1.0, 1e160, 4, prec)[0]
