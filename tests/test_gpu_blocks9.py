"""The 9-point V-cycle on 2 x 2 blocks in LDS against the one-kernel-per-pass
cycle (mg_variant 1), which does the same operations in the same colour order:
stopped after three CG iterations both must hold the same iterate.  The
rounding of the two differs (about 1e-16 per operation); the largest system
here amplifies it by at most its condition number, about 200^2, over three
iterations, hence 1e-9 relative.  Sizes: one tile and less, around the edges of
one tile (64 cells) and of the bottom's depths, several tiles, oblong and odd
grids, one and two sweeps per leg, the consistent and the eliminated
formulation (dx != dy), anisotropic K."""
import numpy as np
import pytest

from helpers import params, pair, rel_err, smooth_c

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1,n2,nu,sweeps,aniso", [
    (5, 5, 2 / 3, 2, False), (7, 40, 1 / 3, 2, False), (33, 33, 2 / 3, 2, False), (63, 64, 2 / 3, 2, False),
    (64, 64, 0.0, 2, True), (65, 66, 2 / 3, 1, False), (100, 50, 2 / 3, 2, False), (108, 117, 1 / 3, 2, True),
    (129, 130, 2 / 3, 1, False), (141, 141, 2 / 3, 2, False), (17, 300, 2 / 3, 2, False), (300, 3, 1 / 3, 2, False),
    (283, 197, 0.5, 2, False),
])
def test_block_cycle_equals_unfused_cycle(gpu_lib, n1, n2, nu, sweeps, aniso):
    from impec2d_amd import capi
    p = params(N1=n1, N2=n2, nu=nu, mu_inj=1 / 20., eps=1e-13, max_iter=3)
    rng = np.random.default_rng(n1 * 1000 + n2)
    shape = (n1 + 4, n2 + 4)
    K11 = np.exp(0.5 * rng.standard_normal(shape))
    K22 = np.exp(0.5 * rng.standard_normal(shape)) if aniso else None
    out = []
    for variant in (0, 1):
        o, g = pair(p, K11, K22, mg_variant=variant, mg_pre=sweeps, mg_post=sweeps)
        g.set_source(o.source())
        g.set_concentration(smooth_c(o))
        try:
            g.pressure_solve()
        except capi.ImpecError as e:
            assert e.code == capi.IMPEC_ENOCONV
        out.append(o.interior(g.get_pressure()).copy())
        g.close()
    assert np.isfinite(out[0]).all()
    assert rel_err(out[0], out[1]) < 1e-9


@pytest.mark.parametrize("n1,n2", [(48, 48), (141, 141), (200, 90)])
def test_block_cycle_iteration_counts(gpu_lib, n1, n2):
    """Run to 1e-10: the same number of iterations (a rounding-sized difference
    of the last residual may cost one) and the same pressure."""
    p = params(N1=n1, N2=n2, nu=2 / 3, mu_res=41.0, mu_inj=1.0, eps=1e-10)
    its, ps = [], []
    for variant in (0, 1):
        o, g = pair(p, mg_variant=variant)
        g.set_source(o.source("circle"))
        g.set_concentration(smooth_c(o))
        n, _ = g.pressure_solve()
        its.append(n)
        ps.append(o.interior(g.get_pressure()).copy())
        g.close()
    assert abs(its[0] - its[1]) <= 1, its
    assert rel_err(ps[0], ps[1]) < 1e-8


@pytest.mark.parametrize("n1,n2,nu,aniso", [(100, 50, 2 / 3, False), (64, 64, 0.5, True), (150, 145, 1 / 3, False),
                                            (9, 5, 2 / 3, False), (3, 3, 2 / 3, True)])
def test_eliminated_formulation_needs_no_search_for_the_constant(gpu_lib, n1, n2, nu, aniso):
    """dx != dy or anisotropic K (the pinned row and column eliminated): the
    preconditioner's constant makes CG start at once.  Without it these solves
    took 21 to 28 iterations, about ten of them for the nearly constant vector; a
    consistent system of the same size takes 10 to 15.  Both cycles agree, as in
    test_block_cycle_iteration_counts."""
    p = params(N1=n1, N2=n2, nu=nu, mu_inj=1 / 20., eps=1e-10)
    rng = np.random.default_rng(n1)
    K11 = np.exp(0.3 * rng.standard_normal((n1 + 4, n2 + 4)))
    K22 = np.exp(0.3 * rng.standard_normal((n1 + 4, n2 + 4))) if aniso else None
    its, ps = [], []
    for variant in (0, 1):
        o, g = pair(p, K11, K22, mg_variant=variant)
        g.set_source(o.source())
        g.set_concentration(smooth_c(o))
        n, _ = g.pressure_solve()
        its.append(n)
        ps.append(o.interior(g.get_pressure()).copy())
        assert g.stats().last_elim_its == n
        g.close()
    assert max(its) <= 20 and abs(its[0] - its[1]) <= 1, its
    assert rel_err(ps[0], ps[1]) < 1e-8


@pytest.mark.parametrize("n1,n2,nu,seed", [(119, 125, 1 / 3, 171), (108, 120, 2 / 3, 199)])
def test_eliminated_formulation_over_many_decades_of_permeability(gpu_lib, n1, n2, nu, seed):
    """Anisotropic white-noise permeability of sigma 4 (over ten decades), with a
    tolerance below the rounding floor: the preconditioner's constant, which
    overshoots there, must not keep a solve from the floor that it reaches with the
    V-cycle alone (0.92 and 0.27 of it; 1.2 times it with the constant throughout)."""
    p = params(N1=n1, N2=n2, nu=nu, x_ub=n1 / n2, avgproc=1, mu_res=10.0, mu_inj=1.0, eps=1e-14, max_iter=3000)
    rng = np.random.default_rng(seed)
    K11, K22 = (np.exp(4.0 * rng.standard_normal((n1 + 4, n2 + 4))) for _ in range(2))
    o, g = pair(p, K11, K22)
    g.set_source(o.source())
    g.set_concentration(smooth_c(o))
    _, rr = g.pressure_solve()
    assert rr <= g.stats().last_relres_floor
    g.close()
