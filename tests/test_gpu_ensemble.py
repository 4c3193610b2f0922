"""Ensembles (impec_ensemble_*): members of different sizes, grids, mobility
ratios and lognormal permeabilities advanced together by batched launches and
graph replays.  Each member must equal, bit for bit, the same problem stepped
alone on its own context with impec_step (which the other GPU tests hold to
the oracle); graph replays and eager launches must agree; chunk heights
picked by the autotuner keep that equality."""
import numpy as np
import pytest

from helpers import gpu_params, pair, params, rel_err, smooth_c
from impec2d_amd import fields
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu

R2 = 2 ** 0.5
# (N1, N2, grid, mobility ratio M, sigma of ln K); grid "diag": injector and
# producer at opposite corners of the unit square, "par": the rotated square
# with four corner wells
MEMBERS = [
    (32, 32, "diag", 10.0, 0.5),
    (48, 40, "par", 30.0, 1.5),
    (64, 64, "diag", 50.0, 2.0),
    (130, 70, "par", 2.0, 1.0),
    (200, 256, "diag", 20.0, 1.0),
]


def _say(*a):
    print(*a, flush=True)


def _member_setup(k, spec, **extra):
    n1, n2, grid, M, sigma = spec
    kw = dict(N1=n1, N2=n2, nu=1.0, eps=1e-10, mu_inj=1.0 / M)
    if grid == "par":
        kw.update(stype=0, x_ub=R2, y_ub=R2)
    p = params(**kw)
    K = fields.lognormal_permeability(n1, n2, sigma=sigma, corr_len=0.05, seed=100 + k,
                                      x_extent=kw.get("x_ub", 1.0), y_extent=kw.get("y_ub", 1.0))
    return p, K


def _run_single(p, K, steps, **extra):
    o, g = pair(p, K, None, **extra)
    q = o.source("one_cell")
    c0 = smooth_c(o, seed=3)
    g.set_source(q)
    g.set_concentration(c0)
    out = []
    t = 0.0
    for _ in range(steps):
        dt = g.step(t)
        t += dt
        out.append((dt, g.stats().last_its, g.get_concentration(), g.get_pressure(), g.get_velocity()))
    g.close()
    return q, c0, out


def _make_ensemble(specs, rows=None, **extra):
    from impec2d_amd import capi
    plist, Ks = [], []
    for k, spec in enumerate(specs):
        p, K = _member_setup(k, spec)
        gp = gpu_params(p, **extra)
        if rows is not None:
            gp.mg_rows = int(rows[k])
        plist.append(gp)
        Ks.append((p, K))
    ens = capi.Ensemble(plist)
    for k, (p, K) in enumerate(Ks):
        o = po.Oracle(p, K, None)   # host-side source and initial state
        m = ens.members[k]
        m.set_permeability(K, None)
        m.set_source(o.source("one_cell"))
        m.set_concentration(smooth_c(o, seed=3))
    return ens, Ks


def _ensemble_steps(ens, steps):
    res = []
    for _ in range(steps):
        dt, its = ens.step()
        res.append((dt.copy(), its.copy(), [(m.get_concentration(), m.get_pressure(), m.get_velocity())
                                             for m in ens.members]))
    return res


@pytest.mark.parametrize("precision,guess", [(0, 0), (1, 1)])
def test_members_equal_single_contexts_bitwise(gpu_lib, precision, guess):
    steps = 3
    _say("ensemble vs single contexts: precision %d guess %d" % (precision, guess))
    ens, Ks = _make_ensemble(MEMBERS, precision=precision, initial_guess=guess)
    res = _ensemble_steps(ens, steps)
    ens.close()
    for k, (p, K) in enumerate(Ks):
        _, _, single = _run_single(p, K, steps, precision=precision, initial_guess=guess)
        for s in range(steps):
            dt_e, its_e, fields_e = res[s][0][k], res[s][1][k], res[s][2][k]
            dt_s, its_s, c_s, p_s, v_s = single[s]
            c_e, p_e, v_e = fields_e
            _say("  member %d step %d: its %d/%d dt %.6e" % (k, s, its_e, its_s, dt_e))
            assert its_e == its_s
            assert dt_e == dt_s
            assert np.array_equal(p_e, p_s)
            assert np.array_equal(v_e, v_s)
            assert np.array_equal(c_e, c_s)


def test_large_member_equal_single_context_bitwise(gpu_lib):
    """A 2048^2 member leaves more partials than one workgroup combines quickly
    (16384 after the CG update): the single context combines them in two
    launches, the ensemble in one workgroup per member, and the two must agree
    bit for bit."""
    steps = 2
    specs = [(2048, 2048, "par", 10.0, 1.0), (64, 48, "diag", 20.0, 1.0)]
    _say("ensemble with a 2048^2 member vs single contexts")
    ens, Ks = _make_ensemble(specs)
    res = _ensemble_steps(ens, steps)
    ens.close()
    for k, (p, K) in enumerate(Ks):
        _, _, single = _run_single(p, K, steps)
        for s in range(steps):
            dt_e, its_e, (c_e, p_e, v_e) = res[s][0][k], res[s][1][k], res[s][2][k]
            dt_s, its_s, c_s, p_s, v_s = single[s]
            _say("  member %d step %d: its %d/%d" % (k, s, its_e, its_s))
            assert its_e == its_s and dt_e == dt_s
            assert np.array_equal(p_e, p_s)
            assert np.array_equal(v_e, v_s)
            assert np.array_equal(c_e, c_s)


@pytest.mark.parametrize("precision", [0, 1])
def test_members_around_the_folded_sums_limit(gpu_lib, precision):
    """A single context folds the sums of its CG passes into their readers up to
    576^2 cells, an ensemble never does: the members' equality holds the folded sums
    to the finishing launches' bits on both sides of that size, and over levels of
    several tiles."""
    _say("ensemble around the folded sums' limit", precision)
    specs = [(576, 576, "diag", 10.0, 0.5), (577, 576, "diag", 10.0, 0.5), (258, 509, "diag", 5.0, 0.5)]
    ens, Ks = _make_ensemble(specs, precision=precision)
    res = _ensemble_steps(ens, 2)
    ens.close()
    for k, (p, K) in enumerate(Ks):
        _, _, single = _run_single(p, K, 2, precision=precision)
        for s in range(2):
            dts, its, fields_e = res[s][0], res[s][1], res[s][2][k]
            dt_s, its_s, c_s, p_s, v_s = single[s]
            assert its[k] == its_s and dts[k] == dt_s
            for a, b in zip(fields_e, (c_s, p_s, v_s)):
                assert np.array_equal(a, b)


def test_members_with_eps_below_rounding_floor(gpu_lib):
    """eps = 1e-15 lies below the FP64 rounding floor of every member's
    system: a member's recursion can stall short of it.  The device-side loop
    sends a stalled member to the residual recheck and its restart rules, and
    the member stops at its floor (or the host finishes it with the member's
    own solve).  Every solve ends at max(eps, floor) within a bounded number
    of iterations, and the fields agree with the same problem stepped alone to
    what two solves stopped at the rounding floor can share (the two loops
    take their restarts at different iterations there, so bitwise equality is
    not expected)."""
    steps = 3
    _say("ensemble with eps 1e-15 (below the rounding floor)")
    specs = MEMBERS[:4]
    ens, Ks = _make_ensemble(specs, eps=1e-15)
    res = _ensemble_steps(ens, steps)
    worst = 0
    for k in range(len(specs)):
        st = ens.members[k].stats()
        assert st.last_relres <= max(1e-15, st.last_relres_floor), (k, st.last_relres, st.last_relres_floor)
    ens.close()
    for k, (p, K) in enumerate(Ks):
        _, _, single = _run_single(p, K, steps, eps=1e-15)
        for s in range(steps):
            its_e = res[s][1][k]
            c_e, p_e, v_e = res[s][2][k]
            _, its_s, c_s, p_s, v_s = single[s]
            ep, ec = rel_err(p_e, p_s), rel_err(c_e, c_s)
            _say("  member %d step %d: its %d/%d, p %.2e c %.2e" % (k, s, its_e, its_s, ep, ec))
            worst = max(worst, its_e)
            assert ep < 1e-8 and ec < 1e-8
    assert worst <= 200   # no run to the iteration limit


def test_graph_replays_match_eager_launches(gpu_lib):
    """The same ensemble stepped with eager launches, with graphs of one CG
    iteration per replay and with graphs of four: identical fields after
    every step (each step replays the iteration graph several times, with the
    host's synchronisation and reads in between)."""
    steps = 3
    runs = {}
    for mode in [("eager", 0, 0), ("graph1", 1, 1), ("graph4", 1, 4)]:
        _say("ensemble launch mode", mode[0])
        ens, _ = _make_ensemble(MEMBERS[:4], precision=1)
        ens.set_graphs(mode[1], mode[2])
        runs[mode[0]] = _ensemble_steps(ens, steps)
        ens.close()
    for name in ("graph1", "graph4"):
        for s in range(steps):
            a, b = runs["eager"][s], runs[name][s]
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
            for fa, fb in zip(a[2], b[2]):
                for x, y in zip(fa, fb):
                    assert np.array_equal(x, y)


def test_autotuned_rows_keep_member_equality(gpu_lib):
    specs = MEMBERS[:3] + [(512, 512, "diag", 20.0, 1.0)]
    ens, Ks = _make_ensemble(specs)
    rows = ens.autotune(reps=2)
    _say("autotuned finest-level chunk rows", rows.tolist())
    assert all(r in (8, 16, 32, 64) for r in rows)
    for k in range(len(specs)):
        for q in range(len(specs)):
            if specs[q][:2] == specs[k][:2]:
                assert rows[q] == rows[k]
    res = _ensemble_steps(ens, 2)
    ens.close()
    for k, (p, K) in enumerate(Ks):
        _, _, single = _run_single(p, K, 2, mg_rows=int(rows[k]))
        for s in range(2):
            assert res[s][1][k] == single[s][1]
            c_e, p_e, v_e = res[s][2][k]
            assert np.array_equal(p_e, single[s][3]) and np.array_equal(c_e, single[s][2])


def test_members_match_oracle(gpu_lib):
    """One member of each grid type against the oracle stepped with the same
    lognormal K: p, u, v, c after 3 steps within 1e-10 (solves at 1e-13)."""
    from impec2d_amd import capi
    specs = [(40, 40, "diag", 10.0, 1.0), (36, 44, "par", 30.0, 1.5), (48, 48, "diag", 3.0, 0.5)]
    plist, setups = [], []
    for k, (n1, n2, grid, M, sigma) in enumerate(specs):
        kw = dict(N1=n1, N2=n2, nu=1.0, eps=1e-13, mu_inj=1.0 / M)
        if grid == "par":
            kw.update(stype=0, x_ub=R2, y_ub=R2)
        p = params(**kw)
        K = fields.lognormal_permeability(n1, n2, sigma=sigma, corr_len=0.05, seed=300 + k,
                                          x_extent=kw.get("x_ub", 1.0), y_extent=kw.get("y_ub", 1.0))
        plist.append(gpu_params(p))
        setups.append((p, K))
    ens = capi.Ensemble(plist)
    refs = []
    for k, (p, K) in enumerate(setups):
        o = po.Oracle(p, K, None)
        q = o.source("one_cell")
        c0 = smooth_c(o, seed=4)
        m = ens.members[k]
        m.set_permeability(K, None)
        m.set_source(q)
        m.set_concentration(c0)
        refs.append((o, q, c0.copy(), o.scalar(), o.velocity()))
    t_ref = [0.0] * len(specs)
    for s in range(3):
        dt, its = ens.step()
        for k, (o, q, c, pr, v) in enumerate(refs):
            st, dtr = o.step(c, pr, v, q, t_ref[k])
            assert st == 0
            t_ref[k] += dtr
            assert abs(dt[k] - dtr) <= 1e-10 * dtr
    for k, (o, q, c, pr, v) in enumerate(refs):
        m = ens.members[k]
        ec = rel_err(o.interior(m.get_concentration()), o.interior(c))
        ep = rel_err(o.interior(m.get_pressure()), o.interior(pr))
        ev = rel_err(m.get_velocity(), v)
        _say("  member %d %s: c %.2e p %.2e v %.2e" % (k, specs[k][2], ec, ep, ev))
        assert ec < 1e-10 and ep < 1e-10 and ev < 1e-10
    ens.close()


def test_full_size_ensemble_invariants(gpu_lib):
    """The benchmark's ensemble at full size: 256 members, sizes uniform from
    {128, 256, 512, 1024}^2, M in [2, 50], sigma in [0.5, 2], both grids,
    mixed precision with the previous-pressure guess, 3 steps.  Permeabilities
    are made transpose-symmetric (geometric mean of K and K^T), so every
    member's concentration must stay symmetric about the diagonal; every
    member keeps mass balance, div v = q and zero wall flux, and its pressure
    solves reach 1e-10."""
    from impec2d_amd import capi
    import bench
    rng = np.random.default_rng(77)
    members = 256
    sizes = rng.choice([128, 256, 512, 1024], members)
    sigmas = rng.uniform(0.5, 2.0, members)
    Ms = rng.uniform(2.0, 50.0, members)
    grids = rng.integers(0, 2, members)
    plist = []
    for k in range(members):
        n, ext = int(sizes[k]), (1.0 if grids[k] == 0 else R2)
        plist.append(capi.default_params(
            N1=n, N2=n, source_type=capi.SRC_DIAGONAL if grids[k] == 0 else capi.SRC_PARALLEL, nu=1.0,
            dim_splitting=capi.SPLIT_PARALLEL, diffusion=0, x_ub=ext, y_ub=ext, mu_res=1.0, mu_inj=1.0 / Ms[k],
            cfl=0.5, eps=1e-10, precision=capi.PREC_MIXED, initial_guess=capi.GUESS_PREVIOUS))
    _say("full-size ensemble: %d members, %d cells" % (members, int(np.sum(sizes.astype(np.int64) ** 2))))
    ens = capi.Ensemble(plist)
    for k in range(members):
        n, ext = int(sizes[k]), (1.0 if grids[k] == 0 else R2)
        K = fields.lognormal_permeability(n, n, sigma=sigmas[k], corr_len=0.05, seed=5000 + k, x_extent=ext,
                                          y_extent=ext)
        K = np.sqrt(K * K.T)
        m = ens.members[k]
        m.set_permeability(np.ascontiguousarray(K), None)
        m.set_source(bench.one_cell_source(n) if grids[k] == 0 else bench.corner_wells_source(n))
    t = np.zeros(members)
    for s in range(3):
        dt, its = ens.step()
        t += dt
        _say("  step %d: CG iterations %d..%d" % (s, its.min(), its.max()))
    worst = dict(mass=0.0, div=0.0, sym=0.0)
    for k in range(members):
        m = ens.members[k]
        st = m.stats()
        # 1e-10, or the FP64 floor of the residual where K spans five decades
        assert st.last_relres <= max(1e-10, st.last_relres_floor), (k, st.last_relres, st.last_relres_floor)
        me = m.mass_error(t[k])
        worst["mass"] = max(worst["mass"], me)
        assert me < 1e-9, (k, me)
        assert m.velocity_boundary_error() == 0.0, k
        de = m.divergence_error()
        worst["div"] = max(worst["div"], de)
        assert de < 1e-6, (k, de)
        c = m.get_concentration()[2:-2, 2:-2]
        sym = np.abs(c - c.T).max() / max(np.abs(c).max(), 1e-300)
        worst["sym"] = max(worst["sym"], sym)
        assert sym < 1e-8, (k, sym)
    _say("  worst mass error %.2e, divergence error %.2e, asymmetry %.2e" % (worst["mass"], worst["div"],
                                                                             worst["sym"]))
    ens.close()
