"""GPU test of the hybrid plan's nodal solve (explicit symmetric inverses with
refinement) against the pivoted Z_L-first FP64 factor of the assembled W, at
the sizes where its kernels change shape: segment and node counts around the
16-row strips, the 64-row tiles and the 64-, 128- and 256-column steps, one
segment, and the route out of it (a zero frequency makes Z_L vanish, so the
nodal solve cannot accept and the pivoted factor answers).

Tolerances. U[inj]: the FP64 form is refined to an estimated 1e-14 and the
mixed one to 1e-10 of |x|, so what remains is the LU's own error, taken at the
1e-9 of the other plan comparisons in FP64 and the 1e-8 bar in the mixed form.
The whole x, relative to its largest entry: 1e-8 (the LU's normwise error at
cond(W) ~ 1e8)."""
import numpy as np
import pytest

import tags_pkg

T = tags_pkg.load()

pytestmark = pytest.mark.gpu


def _routes(kind, taken, left, before):
    """The route counts since `before`: a sample that the solve under test leaves to
    the pivoted factor would be answered by what it is compared with."""
    now = T.route_counts()[kind]
    assert (now[0] - before[0], now[1] - before[1]) == (taken, left)
    return now


def _rod(m):
    rc, e, nodes = T.segment_electrode([0, 0, -0.5], [0.5 * m, 0, -0.5], m, 7e-3)
    return e, nodes


def _grid(vx, vy, ex, ey):
    rc, e, nodes = T.electrode_grid(vx, vy, 0.6 * ex * (vx - 1), 0.6 * ey * (vy - 1), ex, ey, 5e-3,
                                    -0.6)
    return e, nodes


def _compare(e, nodes, f, groups=(0,), mhem=False):
    s = 2j * np.pi * np.asarray(f)
    kap = 2e-3 + s * 12.0 * T.EPS0
    inj = len(nodes) // 2
    sw = T.Sweep(e, nodes)
    if mhem:
        sw.set_formulation(T.FORM_MHEM)
    sw.set_plan(T.PLAN_ZL_FIRST)
    u0, _, x0 = sw.solve(s, kap, inj, T.PREC_FP64, want_x=True)
    sw.set_plan(T.PLAN_HYBRID)
    scale = np.abs(x0).max(axis=1, keepdims=True)
    for g in groups:
        sw.set_batch(g)
        for prec, tol in ((T.PREC_FP64, 1e-9), (T.PREC_MIXED, 1e-8)):
            r0 = T.route_counts()["nodal"]
            u, st, x = sw.solve(s, kap, inj, prec, want_x=True)
            _routes("nodal", len(s), 0, r0)
            assert all(q["info"] == 0 and q["precision_used"] == prec for q in st), (prec, st)
            assert np.max(np.abs(u - u0) / np.abs(u0)) <= tol, (prec, g)
            assert np.max(np.abs(x - x0) / scale) <= 1e-8, (prec, g)
            assert np.array_equal(u, x[:, inj])
    sw.close()


@pytest.mark.parametrize("m", [1, 2, 15, 16, 17, 31, 32, 63, 64, 65, 127, 128, 129, 191])
def test_conductors_at_tile_edges(m):
    _compare(*_rod(m), f=[60.0, 1e4, 3e6], groups=(0, 2))


# (segments, nodes): (10, 10), (262, 239), (635, 580), (705, 636)
@pytest.mark.parametrize("shape", [(2, 2, 3, 2), (7, 5, 5, 4), (9, 8, 5, 5), (11, 8, 4, 5)])
def test_grids_across_the_step_widths(shape):
    _compare(*_grid(*shape), f=[100.0, 2e5])


# around the order from which complex64 takes 256-column steps, and its second step
@pytest.mark.parametrize("m", [299, 300, 321, 511, 513])
def test_conductors_across_wide_steps(m):
    _compare(*_rod(m), f=[1e4, 3e6])


def test_mhem_blocks():
    _compare(*_grid(4, 3, 5, 3), f=[100.0, 1e5, 2e6], mhem=True)


def test_zero_frequency_takes_the_pivoted_factor():
    e, nodes = _rod(20)
    s = np.array([0.0, 2j * np.pi * 1e5])
    kap = 2e-3 + s * 12.0 * T.EPS0
    sw = T.Sweep(e, nodes)
    sw.set_plan(T.PLAN_ZL_FIRST)
    u0, st0 = sw.solve(s, kap, 0, T.PREC_FP64)
    sw.set_plan(T.PLAN_HYBRID)
    for prec in (T.PREC_FP64, T.PREC_MIXED):
        r0 = T.route_counts()["nodal"]
        u, st = sw.solve(s, kap, 0, prec)
        _routes("nodal", 1, 1, r0)
        assert [q["info"] for q in st] == [q["info"] for q in st0]
        ok = np.isfinite(u0)
        assert np.array_equal(np.isfinite(u), ok)
        assert np.all(np.abs(u - u0)[ok] <= 1e-8 * np.abs(u0[ok]))
    sw.close()


@pytest.mark.parametrize("inflight", [1, 4])
def test_a_rejected_sample_leaves_the_others_alone(inflight):
    """Samples around ones that the nodal solve does not accept (zero frequency)
    answer bit for bit as in a call without them, in both forms, one sample a
    group and on one slot or several; the rejected ones as the pivoted plan does
    (1e-9, as the other comparisons with it), whether they share a group or not."""
    e, nodes = _rod(70)
    f = np.array([50.0, 0.0, 3e3, 0.0, 1e5, 0.0, 2e6])
    s = 2j * np.pi * f
    kap = 2e-3 + s * 12.0 * T.EPS0
    z = f == 0
    sw = T.Sweep(e, nodes)
    sw.set_inflight(inflight)
    for prec in (T.PREC_FP64, T.PREC_MIXED):
        sw.set_plan(T.PLAN_ZL_FIRST)
        p = sw.solve(s, kap, 3, prec)[0]
        sw.set_plan(T.PLAN_HYBRID)
        sw.set_batch(1)
        r0 = T.route_counts()["nodal"]
        u, st, x = sw.solve(s, kap, 3, prec, want_x=True)
        _routes("nodal", 4, 3, r0)
        v, sv, y = sw.solve(s[~z], kap[~z], 3, prec, want_x=True)
        assert np.array_equal(u[~z], v) and np.array_equal(x[~z], y)
        assert [q["refine_iters"] for q, r in zip(st, z) if not r] == [q["refine_iters"] for q in sv]
        sw.set_batch(0)
        w = sw.solve(s, kap, 3, prec)[0]
        for got in (u, w):
            assert np.allclose(got[z], p[z], rtol=1e-9, atol=0.0, equal_nan=True)
    sw.close()


def _conductors(rods):
    """Separate straight conductors (start, end, segments), their nodes shuffled."""
    e, nodes = zip(*[T.segment_electrode(a, b, k, 7e-3)[1:] for a, b, k in rods])
    e, nodes = np.concatenate(e), np.concatenate(nodes)
    return e, nodes[np.random.default_rng(len(e)).permutation(len(nodes))]


_RODS = [([0, 0, -0.5], [15, 0, -0.5]), ([0, 20, -0.5], [12, 20, -0.5]), ([30, 0, -0.5], [30, 0, -3.5]),
         ([3, 1, -0.6], [3, 9, -0.6])]


# (segments of each): few and small, past 64 nodes, beyond the 128- and 256-column steps;
# single segments, which a part's root and one more node make up
@pytest.mark.parametrize("counts", [(3, 2), (30, 24), (30, 24, 6), (1, 1, 1, 1), (60, 50, 6, 20),
                                    (20, 150, 9), (210, 90, 12)])
@pytest.mark.parametrize("mhem", [False, True])
def test_separate_conductors(counts, mhem):
    """Several conductors that no segment joins, injected at a root, at another
    node of a part and at the largest part: as one conductor is, and refined in the
    steps that one takes. Without their constants taken out, two rods contract by
    0.03 to 0.1 a step at 60 Hz and the mixed form needs 10 steps and more; one
    conductor of 30 segments needs the three that are always done, a longer one
    at most two more (1e-2 a step is the slowest that the node system is known
    for, 1e-10 the goal)."""
    e, nodes = _conductors([(a, b, k) for (a, b), k in zip(_RODS, counts)])
    f = [60.0, 1e4, 3e6]
    _compare(e, nodes, f, mhem=mhem)
    s = 2j * np.pi * np.asarray(f)
    kap = 2e-3 + s * 12.0 * T.EPS0
    sw = T.Sweep(e, nodes)
    if mhem:
        sw.set_formulation(T.FORM_MHEM)
    for end in ([0, 0, -0.5], [0, 20, -0.5], [12, 20, -0.5]):
        inj = int(np.argmin(np.linalg.norm(nodes - end, axis=1)))
        sw.set_plan(T.PLAN_ZL_FIRST)
        u0, _, x0 = sw.solve(s, kap, inj, T.PREC_FP64, want_x=True)
        sw.set_plan(T.PLAN_HYBRID)
        scale = np.abs(x0).max(axis=1, keepdims=True)
        for prec, tol in ((T.PREC_FP64, 1e-9), (T.PREC_MIXED, 1e-8)):
            u, st, x = sw.solve(s, kap, inj, prec, want_x=True)
            assert np.max(np.abs(u - u0) / np.abs(u0)) <= tol
            assert np.max(np.abs(x - x0) / scale) <= 1e-8
            assert all(q["precision_used"] == prec and q["refine_iters"] <= 5 for q in st), st
    sw.close()


@pytest.mark.parametrize("lanes", [1, 3])
def test_cases_with_rejected_samples_and_separate_conductors(lanes):
    """Many cases over lanes, each lane's solver serving one and several parts in
    turn, with samples that the nodal solve rejects: every case as its own sweep
    gives it, accepted samples bit for bit."""
    f = np.array([50.0, 0.0, 2e4, 1e6])
    s = 2j * np.pi * f
    kap = 2e-3 + s * 12.0 * T.EPS0
    geo = [_rod(20), _conductors([(a, b, k) for (a, b), k in zip(_RODS, (30, 24, 6))]), _rod(90),
           _conductors([(a, b, k) for (a, b), k in zip(_RODS, (3, 2))]), _rod(70)]
    descs = [dict(electrodes=e, nodes=nodes, s=s, kappa=kap, inj_node=1) for e, nodes in geo]
    cs = T.Cases(descs)
    cs.set_lanes(lanes)
    for prec in (T.PREC_FP64, T.PREC_MIXED):
        r0 = T.route_counts()["nodal"]
        got, _ = cs.solve(prec)
        _routes("nodal", 3 * len(geo), len(geo), r0)
        for u, (e, nodes) in zip(got, geo):
            sw = T.Sweep(e, nodes)
            v = sw.solve(s, kap, 1, prec)[0]
            sw.close()
            assert np.array_equal(u[f > 0], v[f > 0])
            assert np.allclose(u, v, rtol=1e-9, atol=0.0, equal_nan=True)
    cs.close()
