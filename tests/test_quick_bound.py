"""The quick score bounds of the 3-way kernels (quick_bound and the host's
constants for it): FP32 cells derived from FP32 marginals, 1/T replaced by
recip_above, log2 by float bits, and the second bound's per-cell curvature.
Emulated in numpy FP32 and held against the oracle's exact K2 and MI: what the
kernel rules a set out with is never above the set's exact badness by more
than the rounding allowance the kernel's threshold already has.
"""
import math

import numpy as np
import pytest

import oracle as O

F = np.float32
U = 2.0 ** -24


def recip_above(t):
    return (np.uint32(0x7F000000) - t.view(np.uint32)).view(F)


def constants(Nc, Nt, score, cells):
    """make_ctx's quick-bound constants."""
    N = Nc + Nt
    qc, qt = Nc / N, Nt / N
    K = max(-math.log1p(-qc) / qc ** 2, -math.log(qc) / qt ** 2) * (1 + 1e-6)
    scale, top, lnw, off = K, -N * (qc * math.log(qc) + qt * math.log(qt)), 0.5 * math.log(2), \
        -cells * 0.5 * math.log(math.pi / 2) * (1 + 1e-6)
    if score == O.MI:
        scale, top, lnw, off = K / (N * math.log(2)), 0.0, 0.0, 0.0
    eta = 57.3 * U * math.sqrt(N)
    kpi = 1 / (2 * qc * qt)
    slope = max(0.0, (-math.log1p(-qc) / qc ** 2 - kpi) / qc, (-math.log(qc) / qt ** 2 - kpi) / qt)
    loss = 3 * eta * math.sqrt(1.125 * (1 + 1.125 * slope / kpi))
    widen = scale / K * (1 + 1e-6) / (1 - loss) * (1 + 1e-5)
    extra = 1e-7 * N + 1.0 if score == O.K2 else 1e-6
    return dict(pi=F(qc), fb=F(scale / (1 - eta) ** 2 * (1 + 1e-5)), top=F(top), lnw=F(lnw * 2.0 ** -23), off=F(off),
                k=F(kpi * widen) if loss < 0.5 else F(1e30), a=F(slope * widen) if loss < 0.5 else F(0), extra=extra)


def fma(a, b, c):
    return (a.astype(np.float64) * np.float64(b) + c.astype(np.float64)).astype(F)


def derive27(base, xy, xz, yz):
    """derive27 in FP32: base [2][2][2], xy [3][2] (rows 00 01, 10 11, 20 21), xz [3][3], yz [2][2]."""
    t = np.zeros((3, 3, 3), F)
    t[:2, :2, :2] = base
    t[:2, :2, 2] = (xy[:2] - t[:2, :2, 0]) - t[:2, :2, 1]
    t[:2, 2, :] = (xz[:2] - t[:2, 0, :]) - t[:2, 1, :]
    t[2, :2, :2] = (yz - t[0, :2, :2]) - t[1, :2, :2]
    t[2, :2, 2] = (xy[2] - t[2, :2, 0]) - t[2, :2, 1]
    t[2, 2, :] = (xz[2] - t[2, 0, :]) - t[2, 1, :]
    return t.reshape(-1)


def quick_bounds(cas, ctl, score):
    """(first, second) lower bounds of the table's badness, as the kernel computes them."""
    cas, ctl = (np.asarray(v, np.int64).reshape(3, 3, 3) for v in (cas, ctl))
    c = constants(int(cas.sum()), int(ctl.sum()), score, 27)

    def marginals(v):
        return [v[:2, :2, :2], v.sum(2)[:, :2], v.sum(1), v.sum(0)[:2, :2]]
    parts_t = [m.astype(F) for m in marginals(cas + ctl)]
    parts_d = [fma(t, -c["pi"], m.astype(F)) for t, m in zip(parts_t, marginals(cas))]
    T, D = derive27(*parts_t), derive27(*parts_d)
    assert (T == (cas + ctl).reshape(-1)).all()             # totals are exact
    t = np.maximum(T, F(1))
    e = (D * recip_above(t)).astype(F)
    s1 = s2 = F(0)
    for i in range(27):
        s1 = F(np.float64(D[i]) * np.float64(e[i]) + np.float64(s1))
        w = F(np.float64(c["a"]) * abs(np.float64(e[i])) + np.float64(c["k"]))
        s2 = F(np.float64(F(D[i] * e[i])) * np.float64(w) + np.float64(s2))
    bits = int((t.view(np.uint32).astype(np.int64) - 0x3F800000).sum())
    assert 0 <= bits < 2 ** 32
    top = np.float64(c["lnw"]) * bits + np.float64(c["top"]) + np.float64(c["off"])
    return top - np.float64(c["fb"]) * s1, top - np.float64(s2), c["extra"]


def test_recip_above_exhaustive():
    for exp in (0, 22):
        t = (np.arange(1 << 23, dtype=np.uint32) + np.uint32((127 + exp) << 23)).view(F)
        p = recip_above(t).astype(np.float64) * t.astype(np.float64)
        assert p.min() >= 1.0 and p.max() <= 1.125


def test_per_cell_curvature_is_an_upper_bound():
    for pi in (0.001, 0.05, 0.2, 0.3, 0.5, 0.62, 0.9, 0.999):
        p = np.linspace(0.0, 1.0, 200001)
        d = p - pi
        p, d = p[np.abs(d) > 1e-6], d[np.abs(d) > 1e-6]
        with np.errstate(divide="ignore", invalid="ignore"):
            kl = np.where(p > 0, p * np.log(p / pi), 0.0) + np.where(p < 1, (1 - p) * np.log((1 - p) / (1 - pi)), 0.0)
        k0, kpi, k1 = -math.log1p(-pi) / pi ** 2, 1 / (2 * pi * (1 - pi)), -math.log(pi) / (1 - pi) ** 2
        a = max(0.0, (k0 - kpi) / pi, (k1 - kpi) / (1 - pi))
        assert (kl <= d * d * (kpi + a * np.abs(d)) * (1 + 1e-9) + 1e-15).all(), pi


@pytest.mark.parametrize("score", [O.K2, O.MI])
def test_quick_bounds_below_exact_scores(score):
    rng = np.random.default_rng(5 + score)
    skipped = 0
    for trial in range(1200):
        kind = trial % 6
        Nc, Nt = (int(x) for x in rng.integers(1, 40 if kind == 4 else 6000, 2))
        if kind == 5:
            Nc, Nt = int(rng.integers(1, 4)), int(rng.integers(1000, 2000000))
        if kind == 3:
            Nc, Nt = (int(x) for x in rng.integers(100000, 4000000, 2))
        p = rng.dirichlet(np.full(27, rng.uniform(0.05, 3.0)))
        q = rng.dirichlet(np.full(27, rng.uniform(0.05, 3.0))) if kind == 1 else p
        if kind == 2:                       # every cell cases or controls only
            m = rng.random(27) < 0.5
            p, q = np.where(m, p, 0) + 1e-300, np.where(m, 0, p) + 1e-300
            p, q = p / p.sum(), q / q.sum()
        cas, ctl = rng.multinomial(Nc, p).astype(np.uint32), rng.multinomial(Nt, q).astype(np.uint32)
        exact = O.score_k2(cas, ctl) if score == O.K2 else -O.score_mi(cas, ctl)
        first, second, extra = quick_bounds(cas, ctl, score)
        assert first <= exact + extra and second <= exact + extra, (trial, first, second, exact, cas, ctl)
        skipped += second > exact - abs(exact) * 0.05 - 0.02
    assert skipped > 120                    # and they are close enough to rule sets out
