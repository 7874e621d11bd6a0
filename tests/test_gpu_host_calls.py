"""GPU tests of the host-pointer calls' routes: the order rule of the field
integrals, the staged copies at their chunk edges, the symmetric inverse (and
the pivoted factorisation that takes over from it) behind the admittance calls,
the nodal solve behind solve_immittance, and the transforms' twiddles."""
import numpy as np
import pytest

import tags_pkg

T = tags_pkg.load()
O = tags_pkg.oracle()

pytestmark = pytest.mark.gpu


def _fields_ref(p, a, b, il, it, sc):
    """One segment, 40 panels of 20 points graded to the closest axis point, in
    extended precision."""
    p, a, b = (np.asarray(v, np.longdouble) for v in (p, a, b))
    d = b - a
    t0 = np.clip(np.dot(p - a, d) / np.dot(d, d), 0, 1)
    x, w = np.polynomial.legendre.leggauss(20)
    br = np.unique(np.concatenate([[0, 1, t0]] + [np.clip(t0 + s * 2.0 ** -np.arange(20.0), 0, 1)
                                                  for s in (-1, 1)]))
    h = np.diff(br)
    t = (br[:-1, None] + 0.5 * h[:, None] * (1 + x)).ravel()
    wt = (0.5 * h[:, None] * w).ravel()
    q = p - (a + t[:, None] * d)
    r = np.linalg.norm(q, axis=1)
    ex = np.exp(-sc["gamma"] * r)
    ks = np.sum(wt * ex / r)
    kf = np.sum((wt * (1 + sc["gamma"] * r) * ex / r ** 3)[:, None] * q, axis=0)
    va = il * ks * d * T.MU0 / T.FOUR_PI
    k4 = T.FOUR_PI * sc["kappa"]
    return it * ks / k4, va, it * kf / k4 - sc["s"] * va


@pytest.mark.parametrize("freq", [1e3, 3e6, 3e7])
def test_field_orders(freq):
    """Distances on both sides of 1, 1.2, 2, 3.5, 8 and 16 lengths, beside, past
    the end of and obliquely to a 1 m segment; |gamma| L 0.008 .. 2.8 (every
    order, and the graded panels; at 300 MHz the rounding of the phase |gamma| r
    alone, up to 2400, passes 1e-13). The rules are chosen for a remainder of 1e-17
    beside the integral: 1e-13 leaves the rounding of 16 terms and of the
    reference."""
    sc = T.soil_scalars(freq, 0.01, 20.0)
    a, b = np.array([0.3, -0.2, -0.5]), np.array([0.3, 0.8, -0.5])
    rc, e = T.populate_electrode(a, b, 5e-3)
    il, it = np.array([[1.2 - 0.4j]]), np.array([[0.3 + 0.9j]])
    pts = []
    for r in (0.05, 0.999, 1.001, 1.199, 1.201, 1.999, 2.001, 3.49, 3.51, 7.99, 8.01, 15.9, 16.1, 90.0):
        pts += [[0.3 + r, 0.3, -0.5], [0.3, 0.8 + r, -0.5], [0.3, -0.2, -0.5 - r],
                [0.3 + 0.6 * r, 0.8 + 0.64 * r, -0.5 + 0.48 * r]]
    got = T.fields(pts, e, il, it, sc["gamma"], sc["s"], sc["kappa"])
    for j, p in enumerate(np.array(pts)):
        for g, ref in zip(got, _fields_ref(p, a, b, il[0, 0], it[0, 0], sc)):
            assert np.max(np.abs(g[j, 0] - ref)) <= 1e-13 * np.max(np.abs(ref)), (p, g[j, 0], ref)


@pytest.mark.parametrize("np_,m,nrhs", [(1, 1, 1), (1, 257, 2), (3, 600, 5), (2100, 20, 3)])
def test_field_ranges_add_up(np_, m, nrhs):
    """Ranges of segments and groups of right-hand sides against sums over the
    segments one at a time (rounding of m terms: 1e-13)."""
    rng = np.random.default_rng(np_ + m)
    rc, e, nodes = T.segment_electrode([0, 0, -0.5], [0.5 * m, 0, -0.5], m, 7e-3)
    pts = np.column_stack([rng.uniform(-2, 0.5 * m + 2, np_), rng.uniform(1, 9, np_), np.zeros(np_)])
    il, it = (rng.standard_normal((nrhs, m)) + 1j * rng.standard_normal((nrhs, m)) for _ in range(2))
    sc = T.soil_scalars(1e5, 0.01, 10.0)
    got = T.fields(pts, e, il, it, sc["gamma"], sc["s"], sc["kappa"])
    sel = range(0, m, max(1, m // 40))
    part = [sum(x) for x in zip(*[T.fields(pts, e[j:j + 1], il[:, j:j + 1], it[:, j:j + 1], sc["gamma"],
                                           sc["s"], sc["kappa"]) for j in sel])]
    mask = np.zeros(m)
    mask[list(sel)] = 1
    want = T.fields(pts, e, il * mask, it * mask, sc["gamma"], sc["s"], sc["kappa"])
    for w, p, g in zip(want, part, got):
        assert np.max(np.abs(w - p)) <= 1e-13 * max(np.max(np.abs(p)), np.max(np.abs(g)))


@pytest.mark.parametrize("m", [1, 5, 64, 511, 513, 725])
def test_impedance_rows_and_chunks(m):
    """The packed triangle and its 4 MiB chunks (m = 725: a chunk ends inside a
    row): other entries untouched, images added, zl == zt as the reference
    writes it; against the device-pointer form's formulas on separate arrays."""
    rc, e, nodes = T.segment_electrode([0, 0, -0.5], [0.5 * m, 0, -0.5], m, 7e-3)
    img = T.images_of(e)
    sc = T.soil_scalars(2e5, 0.01, 10.0)
    args = (sc["gamma"], sc["s"], 1.0, sc["kappa"])
    fill = 3.0 - 2.0j
    zl, zt, al = (np.full(m * m, fill) for _ in range(3))
    assert T.calculate_impedances(zl, zt, e, *args) == 0
    assert T.calculate_impedances(al, al, e, *args) == 0
    up = np.triu(np.ones((m, m), bool)).ravel()
    dg = np.eye(m, dtype=bool).ravel()
    for z in (zl, zt, al):
        assert np.all(z[~up] == fill) and not np.any(z[up] == fill)
    assert np.array_equal(al[dg], zt[dg]) and np.array_equal(al[up & ~dg], zl[up & ~dg])
    i, k = np.triu_indices(m)
    pick = np.unique(np.linspace(0, len(i) - 1, 40).astype(int))
    rl, rt = O.z_entries(e, img, np.column_stack([i, k])[pick], sc, rel_tol=1e-11, threads=8)
    l0, t0, a0 = zl.copy(), zt.copy(), al.copy()
    assert T.impedances_images(zl, zt, e, img, *args, sc["ref_l"], sc["ref_t"]) == 0
    assert T.impedances_images(al, al, e, img, *args, sc["ref_l"], sc["ref_t"]) == 0
    for z in (zl, zt, al):
        assert np.all(z[~up] == fill)
    at = (i * m + k)[pick]
    assert np.all(np.abs(zl[at] - rl) <= 1e-9 * np.abs(rl) + 1e-14 * np.abs(rl).max())
    assert np.all(np.abs(zt[at] - rt) <= 1e-9 * np.abs(rt) + 1e-14 * np.abs(rt).max())
    both = a0 + (zl - l0) + (zt - t0)
    assert np.all(np.abs(al - both)[up] <= 1e-14 * np.abs(both[up]) + 1e-15 * np.abs(both[up]).max())


def _symmetric(m, seed, definite):
    rng = np.random.default_rng(seed)
    r = rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))
    return (r + r.T) / 2 + (4 * np.sqrt(m) * np.eye(m) if definite else 0)


@pytest.mark.parametrize("m", [1, 2, 63, 64, 65, 128, 129, 200])
@pytest.mark.parametrize("kind", ["dominant", "indefinite", "zero_pivot", "zero_block"])
def test_symmetric_inverse_and_its_fallback(m, kind):
    """solve_admittance and calculate_yla_ytb on matrices that the inverse
    without row exchanges takes, on ones whose growth without them its checks
    have to see, on ones with an exactly zero first pivot (which the 2 x 2 pivots
    take) and with a zero first 2 x 2 block (which nothing without row exchanges
    does): against numpy, 1e-14 of the largest entry times cond (a stable solve's
    normwise bound at these orders, with a factor of about 100 to spare). The
    counts tell that the first kind stays on the route and the last leaves it."""
    if kind == "zero_pivot" and m == 1:
        pytest.skip("a singular 1 x 1 matrix")
    a = _symmetric(m, 5 + m, kind == "dominant")
    if kind == "zero_block" and m < 5:
        pytest.skip("a singular matrix")
    if kind == "zero_pivot":
        a[0, 0] = 0.0
    if kind == "zero_block":
        a[:2, :2] = 0.0
    routes = T.route_counts()
    cond = np.linalg.cond(a)
    rng = np.random.default_rng(m)
    b = rng.standard_normal(m) + 1j * rng.standard_normal(m)
    x = b.copy()
    assert T.solve_admittance(a.T.ravel().copy(), x, m) == 0
    ref = np.linalg.solve(a, b)
    assert np.abs(x - ref).max() <= 1e-14 * cond * np.abs(ref).max()
    n = max(1, m // 2)
    A, B = (rng.standard_normal((m, n)) + 0j for _ in range(2))
    zl, zt = (np.tril(z).T.ravel().copy() for z in (a, _symmetric(m, 99, True)))
    yla, ytb = np.zeros(m * n, complex), np.zeros(m * n, complex)
    assert T.calculate_yla_ytb(yla, ytb, zl, zt, A.T.ravel().copy(), B.T.ravel().copy(), m, n) == 0
    inv = np.linalg.inv(a)
    tol = 1e-14 * cond * np.abs(inv).max()
    assert np.abs(yla.reshape(n, m).T - inv @ A).max() <= tol * np.abs(A).sum(0).max()
    got = zl.reshape(m, m).T
    assert np.abs(np.tril(got) - np.tril(inv)).max() <= tol
    assert np.all(got[np.triu_indices(m, 1)] == 0)
    if kind in ("dominant", "zero_block"):
        for call in ("symmetric", "admittance"):
            was, now = routes[call], T.route_counts()[call]
            assert (now[0] - was[0], now[1] - was[1]) == ((1, 0) if kind == "dominant" else (0, 1))


def test_solve_immittance_structure():
    """The system of the drop-in fills by the nodal solve, and one that is not
    an immittance matrix (a node-to-node entry) by the pivoted factor, both with
    a full right-hand side, against numpy on the same W (1e-9: cond ~ 1e5)."""
    rc, e, nodes = T.electrode_grid(3, 4, 7.0, 9.0, 4, 3, 5e-3, -0.6)
    m, n = len(e), len(nodes)
    N = n + 2 * m
    sc = T.soil_scalars(4e5, 2e-3, 12.0)
    zl, zt = np.zeros(m * m, complex), np.zeros(m * m, complex)
    T.calculate_impedances(zl, zt, e, sc["gamma"], sc["s"], 1.0, sc["kappa"])
    W = np.full(N * N, 7.0 + 0j)
    assert T.fill_incidence_imm(W, e, nodes) == 0
    assert T.fill_impedance_imm(W, zl, zt, m, n) == 0
    ao = np.zeros(m * n, complex), np.zeros(m * n, complex)
    O.fill_incidence_adm(e, nodes, *ao)
    A, B = (x.reshape(n, m).T for x in ao)
    dense = W.reshape(N, N).T
    assert np.array_equal(dense[n:n + m, :n], A) and np.array_equal(dense[n + m:, :n], B)
    assert np.array_equal(dense[:n, n:], dense[n:, :n].T)
    assert not np.any(dense[:n, :n]) and not np.any(dense[n:n + m, n + m:])
    rng = np.random.default_rng(1)
    b = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    for change in (False, True):
        if change:
            W[1] = 0.25  # entry (1, 0)
        low = np.tril(W.reshape(N, N).T)
        full = low + np.tril(low, -1).T
        x = b.copy()
        keep = W.copy()
        was = T.route_counts()["immittance"]
        assert T.solve_immittance(W, x, m, n) == 0
        now = T.route_counts()["immittance"]
        assert (now[0] - was[0], now[1] - was[1]) == ((0, 1) if change else (1, 0))
        assert np.array_equal(W, keep)
        ref = np.linalg.solve(full, b)
        assert np.abs(x - ref).max() <= 1e-9 * np.abs(ref).max()


@pytest.mark.parametrize("nt", [2, 3, 5, 64, 100, 1001, 4096])
def test_transform_twiddles(nt):
    """Forward and back against numpy's FFT with the same weights (rounding of
    the sums: 1e-12 of the largest value)."""
    rng = np.random.default_rng(nt)
    f = rng.standard_normal((3, nt))
    tmax = 1e-4
    g, s = T.laplace_trans(f, tmax)
    c, dt = np.log(float(nt) ** 2) / tmax, tmax / (nt - 1)
    k = np.arange(nt)
    ref = np.fft.rfft(f * dt * np.exp(-c * k * dt), axis=-1)
    assert np.abs(g - ref).max() <= 1e-12 * np.abs(ref).max()
    h = np.fft.irfft(g, nt, axis=-1) * nt
    back = T.inv_laplace_trans(g, s, tmax, nt)
    scale = np.exp(c * k * dt) / (nt * dt)
    assert np.max(np.abs(back - h * scale) / scale) <= 1e-12 * np.abs(h).max()


@pytest.mark.parametrize("nt", [7, 1001, 9999])
def test_transform_twiddles_are_rounded_once(nt):
    """The table's entries themselves: the direct sum of an impulse at sample 1
    of height f is f v w^k, v its weight, exactly w^k where f v rounds to a power
    of two (one of the neighbouring f does; sample k = 0 shows which). Against
    extended-precision cosines and sines: 0.505 ulp, a correct rounding and what
    the reference's own 64-bit mantissa and the angle's leave open."""
    tmax = 1e-4
    c, dt = np.log(float(nt) ** 2) / tmax, tmax / (nt - 1)
    f0 = 2.0 ** 10 / (dt * np.exp(-c * dt))
    f = np.zeros((41, nt))
    f[:, 1] = f0 * (1.0 + np.arange(-20, 21) * 2.0 ** -52)
    g, s = T.laplace_trans(f, tmax)
    exact = np.nonzero(g[:, 0] == 2.0 ** 10)[0]
    assert len(exact) > 0
    w = g[exact[0]] * 2.0 ** -10
    # the angle less the nearest multiple q of a quarter turn, so that its rounding
    # is relative: pi num / (4 nt)
    k = np.arange(len(w))
    q = (8 * k // nt + 1) // 2
    x = np.longdouble("3.14159265358979323846264338327950288") * (8 * k - 2 * q * nt) / (4 * nt)
    cs, sn = np.cos(x), np.sin(x)
    re = np.choose(q % 4, [cs, -sn, -cs, sn])
    im = np.choose(q % 4, [-sn, -cs, sn, cs])
    for got, ref in ((w.real, re), (w.imag, im)):
        ulp = np.spacing(np.abs(ref.astype(float)))
        assert np.max(np.abs(got - ref) / ulp) <= 0.505


def _failing(call, needed):
    """call() with its nth device allocation failing, n = 1, 2, .. until it has no
    more: an error where the call cannot do without it (the first `needed`), the
    answer from the pivoted route otherwise; and the answer again afterwards."""
    L = T.lib()
    n = 0
    while True:
        n += 1
        L.tags_fail_allocation(n)
        rc = call()
        left = L.tags_fail_allocation(0)
        if left:
            break
        assert rc == (0 if n > needed else -100), (n, rc)
    assert rc == 0 and call() == 0
    return n - 1


def test_calls_without_room_for_their_inverses():
    """The symmetric inverses and the nodal solve need device memory beside what
    the pivoted factorisation takes: where it does not fit, that one answers."""
    m, n = 70, 50
    rng = np.random.default_rng(3)
    zl0, zt0 = _symmetric(m, 1, True), _symmetric(m, 2, True)
    A, B = (rng.standard_normal((m, n)) + 0j for _ in range(2))
    ref = np.linalg.solve(zl0, A), np.linalg.solve(zt0, B)
    pats = [np.tril(z).T.ravel() for z in (zl0, zt0)]

    def yla_ytb():
        zl, zt = (p.copy() for p in pats)
        out = np.zeros(m * n, complex), np.zeros(m * n, complex)
        rc = T.calculate_yla_ytb(*out, zl, zt, A.T.ravel().copy(), B.T.ravel().copy(), m, n)
        if rc == 0:
            for o, r in zip(out, ref):
                assert np.abs(o.reshape(n, m).T - r).max() <= 1e-12 * np.abs(r).max()
            for z, z0 in ((zl, zl0), (zt, zt0)):
                inv = np.linalg.inv(z0)
                got = z.reshape(m, m).T
                assert np.abs(np.tril(got) - np.tril(inv)).max() <= 1e-12 * np.abs(inv).max()
        return rc

    b = rng.standard_normal(m) + 1j * rng.standard_normal(m)

    def admittance():
        x = b.copy()
        rc = T.solve_admittance(zl0.T.ravel().copy(), x, m)
        if rc == 0:
            assert np.abs(x - np.linalg.solve(zl0, b)).max() <= 1e-12 * np.abs(x).max()
        return rc

    rc, e, nodes = T.electrode_grid(3, 4, 7.0, 9.0, 4, 3, 5e-3, -0.6)
    me, ne = len(e), len(nodes)
    N = ne + 2 * me
    sc = T.soil_scalars(4e5, 2e-3, 12.0)
    zl, zt, W = (np.zeros(k, complex) for k in (me * me, me * me, N * N))
    T.calculate_impedances(zl, zt, e, sc["gamma"], sc["s"], 1.0, sc["kappa"])
    T.fill_incidence_imm(W, e, nodes)
    T.fill_impedance_imm(W, zl, zt, me, ne)
    low = np.tril(W.reshape(N, N).T)
    c = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    y = np.linalg.solve(low + np.tril(low, -1).T, c)

    def immittance():
        x = c.copy()
        rc = T.solve_immittance(W, x, me, ne)
        if rc == 0:
            assert np.abs(x - y).max() <= 1e-9 * np.abs(y).max()
        return rc

    # the arrays themselves and, for the inverses, A and B in row order
    assert _failing(yla_ytb, 4) > 4
    assert _failing(admittance, 2) > 2
    assert _failing(immittance, 2) > 2


def test_admittance_size_limit():
    """65,536 nodes or more stay refused, whichever route would take them."""
    m, n = 1, 65536
    a, b, y, z = (np.ones(m * n, complex) for _ in range(4))
    assert T.calculate_yla_ytb(y, z, np.ones(1, complex), np.ones(1, complex), a, b, m, n) == -13


@pytest.mark.parametrize("counts", [(8, 5), (4, 40, 30)])
def test_solve_immittance_of_separate_conductors(counts):
    """Conductors that no segment joins, a full right-hand side, against numpy on
    the same W (1e-9: cond ~ 1e5)."""
    rods = [T.segment_electrode([0, 7 * k, -0.5 - k], [3 + c, 7 * k, -0.5 - k], c, 7e-3)[1:]
            for k, c in enumerate(counts)]
    e, nodes = (np.concatenate(v) for v in zip(*rods))
    m, n = len(e), len(nodes)
    N = n + 2 * m
    sc = T.soil_scalars(4e5, 2e-3, 12.0)
    zl, zt, W = (np.zeros(k, complex) for k in (m * m, m * m, N * N))
    T.calculate_impedances(zl, zt, e, sc["gamma"], sc["s"], 1.0, sc["kappa"])
    assert T.fill_incidence_imm(W, e, nodes) == 0 and T.fill_impedance_imm(W, zl, zt, m, n) == 0
    low = np.tril(W.reshape(N, N).T)
    rng = np.random.default_rng(m)
    b = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    x = b.copy()
    was = T.route_counts()["immittance"]
    assert T.solve_immittance(W, x, m, n) == 0
    assert T.route_counts()["immittance"] == (was[0] + 1, was[1])
    ref = np.linalg.solve(low + np.tril(low, -1).T, b)
    assert np.abs(x - ref).max() <= 1e-9 * np.abs(ref).max()


@pytest.mark.parametrize("gamma", [np.inf, 1e30 + 1e30j, 1e20j, complex(np.nan, 1.0), complex(0.1, np.inf)])
def test_gamma_without_end_of_panels(gamma):
    """A gamma that is infinite, not a number, or so large that its panels could
    not be told from each other: NaN, and at once."""
    rc, e, nodes = T.segment_electrode([0, 0, -0.5], [2, 0, -0.5], 4, 7e-3)
    pts = np.array([[0.3, 0.4, 0.0], [9.0, 2.0, 0.0]])
    il = it = np.ones((1, 4), complex)
    for v in T.fields(pts, e, il, it, gamma, 1j, 1e-3 + 0j):
        assert np.all(np.isnan(v))
    zl, zt = np.zeros(16, complex), np.zeros(16, complex)
    assert T.calculate_impedances(zl, zt, e, gamma, 1j, 1.0, 1e-3 + 0j, integration_type=T.INTG_SINGLE) == 0
    off = np.triu(np.ones((4, 4), bool), 1).ravel()
    assert np.all(np.isnan(zt[off])) and np.all(np.isfinite(zt[::5]))
