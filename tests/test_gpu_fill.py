"""GPU test of the sweep's impedance fill: over the range of its classes by |gamma|
times the longest segment (13 to 32 Chebyshev terms up to 7.3) and the direct rule
beyond them, on a geometry with touching segments (in line, at a right angle, at 10
degrees, of very different lengths), segments closer than two lengths down to a
tenth of one, far ones, and images of shallow segments. Against the oracle's
adaptive integrals (relative tolerance 1e-11): 1e-9 of each entry, the bar of the
assembly tests. Far pairs against extended precision: 2e-14. Groups of several
samples against single ones: 1e-12 over tiles and sample ranges, bit for bit where
every class meets every other."""
import numpy as np
import pytest

import tags_pkg

T = tags_pkg.load()
O = tags_pkg.oracle()

pytestmark = pytest.mark.gpu


def _geometry():
    d = -0.3
    a = np.deg2rad(10.0)
    chain = [(0, 0, d), (1, 0, d), (2, 0, d), (2, 1, d), (2 + np.cos(a), 1 + np.sin(a), d)]
    segs = [(chain[i], chain[i + 1]) for i in range(4)]
    segs += [((2, 1, d), (3, 1, d))]                       # 10 degrees beside the chain's last
    segs += [((0, 0, d), (0, 0, d - 0.02))]                # fifty times shorter, touching
    segs += [((0, 0.1, d), (1, 0.1, d)), ((0, 0.7, d), (1, 0.7, d)), ((0.2, 1.9, d), (1.1, 1.9, d))]
    segs += [((40, 30, d), (41, 30, d)), ((7, -3, d - 2), (7.5, -3.5, d - 2.5))]
    e = np.zeros(len(segs), T.ELECTRODE_DTYPE)
    for i, (p, q) in enumerate(segs):
        rc, one = T.populate_electrode(p, q, 5e-3)
        e[i] = one[0]
    ends = np.concatenate([e["start_point"], e["end_point"]])
    nodes = np.unique(np.round(ends, 9), axis=0)
    return e, nodes


# |gamma| times the longest segment (1 m) in every class of the moment rule (they end
# at 0.5, 1, 2, 3.7 and 7.3, or where gamma's real part is too large: here at 5) and in
# the direct rule
@pytest.mark.parametrize("glen", [0.02, 0.37, 0.39, 0.7, 1.12, 1.14, 3.6, 3.8, 4.9, 7.2, 7.4, 12.0])
def test_fill_terms_vs_oracle(glen):
    e, nodes = _geometry()
    m, n = len(e), len(nodes)
    # gamma^2 = s mu0 kappa with s = j w, kappa = sigma + s eps: equal conduction
    # and displacement currents, so that both parts of gamma count
    w = glen * np.sqrt(1.0 / (np.sqrt(2.0) * T.MU0 * 15.0 * T.EPS0))
    f = w / (2 * np.pi)
    sc = O.soil_scalars(f, w * 15.0 * T.EPS0, 15.0)
    assert abs(abs(sc["gamma"]) - glen) < 1e-9 * glen
    i, k = np.triu_indices(m)
    pairs = np.column_stack([i, k])
    zl, zt = O.z_entries(e, O.images_of(e), pairs, sc, rel_tol=1e-11, threads=8)
    sw = T.Sweep(e, nodes)
    got = [-sw.assemble_entries(sc["s"], sc["kappa"], o + i, o + k) for o in (n, n + m)]
    low = [-sw.assemble_entries(sc["s"], sc["kappa"], o + k, o + i) for o in (n, n + m)]
    sw.close()
    for g, l, ref in zip(got, low, (zl, zt)):
        err = np.abs(g - ref)
        # entries e^{-|Re gamma| r} below the oracle's absolute floor are left out
        assert np.all(err <= 1e-9 * np.abs(ref) + 1e-13 * np.abs(ref).max()), err.max()
        assert np.array_equal(g, l)


@pytest.mark.parametrize("m,nf", [(1, 3), (16, 5), (17, 1), (33, 70), (150, 9), (256, 9), (257, 9)])
def test_group_fill_matches_single_samples(m, nf):
    """Tiles and sample ranges of a group: U[inj] of a sweep solved in one group
    and one sample at a time."""
    rc, e, nodes = T.segment_electrode([0, 0, -0.5], [0.5 * m, 0, -0.5], m, 7e-3)
    s = 2j * np.pi * 10.0 ** np.linspace(2, 7.5, nf)
    kap = 5e-3 + s * 10.0 * T.EPS0
    sw = T.Sweep(e, nodes)
    res = []
    for b in (0, 1):
        sw.set_batch(b)
        res.append(sw.solve(s, kap, 0, T.PREC_FP64)[0])
    sw.close()
    assert np.max(np.abs(res[0] - res[1]) / np.abs(res[1])) <= 1e-12


def _unit_integral(S, R, g):
    """int int e^{-g r} / r over the unit square in extended precision: 24-point
    Gauss rules on two panels a side (a segment apart or more: below 1e-17)."""
    x, w = np.polynomial.legendre.leggauss(24)
    x, w = (x.astype(np.longdouble) + 1) / 4, w.astype(np.longdouble) / 4
    # one Newton step on P_24 from the 64-bit nodes, and their weights
    z = 4 * x - 1
    p0, p1 = np.ones_like(z), np.zeros_like(z)
    for k in range(1, 25):
        p0, p1 = ((2 * k - 1) * z * p0 - (k - 1) * p1) / k, p0
    dp = 24 * (z * p0 - p1) / (z * z - 1)
    z = z - p0 / dp
    p0, p1 = np.ones_like(z), np.zeros_like(z)
    for k in range(1, 25):
        p0, p1 = ((2 * k - 1) * z * p0 - (k - 1) * p1) / k, p0
    dp = 24 * (z * p0 - p1) / (z * z - 1)
    x, w = (z + 1) / 4, 2 / ((1 - z * z) * dp * dp) / 4
    t, wt = np.concatenate([x, x + np.longdouble(0.5)]), np.concatenate([w, w])
    a, b, c, d = (np.asarray(v, np.longdouble) for v in (*S, *R))
    p, q = a + t[:, None] * (b - a), c + t[:, None] * (d - c)
    r = np.sqrt(((p[:, None] - q[None]) ** 2).sum(axis=2))
    f = np.exp(-g * r) / r
    return (wt[:, None] * wt[None] * f).sum()


# gamma = (1 + 0 j or 1 j) re, exactly: its square is kappa with s = 1 and s mu = 1
@pytest.mark.parametrize("re,im", [(2.0, 0), (3.625, 0), (5.0, 0), (7.25, 0), (1.75, 1), (2.5, 1),
                                   (3.5, 1), (4.9375, 1), (6.0, 1)])
def test_fill_keeps_the_direct_rules_digits(re, im):
    """Far pairs (3 to 20 lengths) of 40 segments of 0.3 to 1 m in random
    directions 12 m deep, with their images, on all sides of the moment rule's
    limits. Against extended precision: 2e-14 of both parts' sizes. (The direct
    rule's rounding and remainder stay below 1e-14 there, largest at |gamma| = 7,
    where the phase of the farthest pair is 140. Below |gamma| = 1 the remainder of
    its orders, not rounding, decides: up to 2.5e-12.)"""
    rng = np.random.default_rng(11)
    m, depth = 40, 12.0
    c = rng.uniform(-7, 7, (m, 3))
    d = rng.standard_normal((m, 3))
    d *= rng.uniform(0.15, 0.5, (m, 1)) / np.linalg.norm(d, axis=1, keepdims=True)
    d[0] *= 0.5 / np.linalg.norm(d[0])
    e = np.zeros(m, T.ELECTRODE_DTYPE)
    for i in range(m):
        e[i] = T.populate_electrode(c[i] - d[i] - [0, 0, depth], c[i] + d[i] - [0, 0, depth], 5e-3)[1][0]
    nodes = np.concatenate([e["start_point"], e["end_point"]])
    g = re * (1 + im * 1j)
    kap = 2j * re * re if im else re * re + 0j
    mur = [v for v in 1 / T.MU0 + np.arange(-4, 5) * np.spacing(1 / T.MU0) if T.MU0 * v == 1.0][0]
    pairs = [(i, k) for i in range(m) for k in range(i) if np.linalg.norm(c[i] - c[k]) >= 4.0]
    pairs = [pairs[j] for j in rng.choice(len(pairs), 60, replace=False)]
    n = len(nodes)
    i, k = np.array(pairs).T
    sw = T.Sweep(e, nodes)
    got = -sw.assemble_entries(1.0, kap, n + m + i, n + m + k, mur=mur)
    sw.close()
    img = T.images_of(e)
    kl = np.clongdouble(kap)
    eps = np.longdouble(T.EPS0)
    for z, (p, q) in zip(got, pairs):
        d, r = (_unit_integral((e[q]["start_point"], e[q]["end_point"]),
                               (x[p]["start_point"], x[p]["end_point"]), np.clongdouble(g))
                for x in (e, img))
        r *= (kl - eps) / (kl + eps)
        err = abs(z * np.longdouble(T.FOUR_PI) * kl - (d + r))
        assert err <= 2e-14 * (abs(d) + abs(r)), (p, q, float(err / (abs(d) + abs(r))))


@pytest.mark.parametrize("m", [9, 17, 257])
def test_a_sample_does_not_see_its_group(m):
    """Samples of every class of the moment rule and of the direct one, in rising
    and in shuffled order, solved in one group, in groups of three and one at a
    time, on one slot and several: the same bits, and W alone the same as W in any
    company (through x)."""
    rc, e, nodes = T.segment_electrode([0, 0, -0.5], [3.0 * m, 0, -0.5], m, 7e-3)
    f = np.concatenate([[50.0], 10.0 ** np.linspace(4, 8, 33)])
    s = 2j * np.pi * f
    kap = 1e-3 + s * 10.0 * T.EPS0
    z = np.abs(np.sqrt(s * T.MU0 * kap)) * 3.0
    assert [np.sum((z > a) & (z <= b)) > 0 for a, b in
            ((0, 0.5), (0.5, 1), (1, 2), (2, 3.7), (3.7, 7.3), (7.3, 1e9))] == [True] * 6
    mix = np.random.default_rng(m).permutation(len(f))
    sw = T.Sweep(e, nodes)
    for prec in (T.PREC_FP64, T.PREC_MIXED):
        ref = None
        for batch, inflight, order in ((1, 1, np.arange(len(f))), (0, 4, np.arange(len(f))),
                                       (0, 1, mix), (3, 2, mix)):
            sw.set_batch(batch)
            sw.set_inflight(inflight)
            u, st, x = sw.solve(s[order], kap[order], 0, prec, want_x=True)
            assert all(q["precision_used"] == prec for q in st)
            back = np.argsort(order)
            if ref is None:
                ref = x[back]
            assert np.array_equal(x[back], ref)
    sw.close()
