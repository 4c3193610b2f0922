"""The bottom of the 5-point V-cycle reads coefficients that are formed once per
solve.  Those of an earlier solve must not be left over: a context that has
solved for another concentration and permeability gives bit for bit the pressure
and the iteration count of a fresh one.  And the solution is that of the legs run
down to the coarsest level (mg_variant 2), to the tolerance times the condition
number (about 260^2 at the largest size).  Sizes: a first level of each depth
(3 to 64 cells a side), ragged and oblong levels, a coarsest level of 1 x 2, 2 x 1
and 2 x 2 cells; both face averages, one and two sweeps, both cycles."""
import numpy as np
import pytest

from helpers import params, pair, random_c, rel_err, smooth_c

pytestmark = pytest.mark.gpu

SIZES = [(5, 5), (9, 130), (16, 16), (33, 20), (40, 7), (65, 63), (128, 128), (128, 3), (129, 66), (257, 131)]
EPS = 1e-11


def _solve(n1, n2, avg, variant, sweeps, precision, used=False):
    p = params(N1=n1, N2=n2, nu=1.0, avgproc=avg, mu_inj=1 / 20., eps=EPS)
    rng = np.random.default_rng(n1 * 1000 + n2)
    K = np.exp(0.5 * rng.standard_normal((n1 + 4, n2 + 4)))
    o, g = pair(p, K, mg_variant=variant, mg_pre=sweeps, mg_post=sweeps, precision=precision)
    g.set_source(o.source())
    if used:
        g.set_permeability(np.exp(0.5 * rng.standard_normal(K.shape)))
        g.set_concentration(random_c(o, seed=3))
        g.pressure_solve()
        g.set_permeability(K)
    g.set_concentration(smooth_c(o))
    its, rr = g.pressure_solve()
    out = o.interior(g.get_pressure()).copy()
    g.close()
    assert rr <= EPS
    return out, its


@pytest.mark.parametrize("avg,sweeps,precision", [(0, 1, 0), (1, 2, 0), (0, 2, 1)])
@pytest.mark.parametrize("n1,n2", SIZES)
def test_bottom_coefficients_are_this_solves(gpu_lib, n1, n2, avg, sweeps, precision):
    a, ia = _solve(n1, n2, avg, 0, sweeps, precision)
    b, ib = _solve(n1, n2, avg, 0, sweeps, precision, used=True)
    assert ia == ib and np.array_equal(a, b)
    assert rel_err(a, _solve(n1, n2, avg, 2, sweeps, precision)[0]) < EPS * 260 ** 2
