"""Cells of zero permeability with the mean-concentration average: a mobility of
zero on both sides of a face makes a zero face, on every level of the cycle, and
a cell of four zero faces stays out of the solve.  The region covers whole coarse
cells down to 1/16 of the grid, a barrier one cell wide makes single zero faces,
and both lie away from the wells and the pinned cell.  The one-kernel-per-pass
cycle (mg_variant 1) forms every face by itself and is the reference: each solves
to a relative residual of 1e-11, so the pressures agree to that times the
condition number (about 200^2 times the mobility ratio of 20 at the largest
size), 1e-5, wherever the pressure is determined, that is outside the region.
Sizes: the first level of the bottom kernel, tile legs above it, several tiles."""
import numpy as np
import pytest

from tests.helpers import pair, params, smooth_c

pytestmark = pytest.mark.gpu

EPS = 1e-11


def _solve(n1, n2, nu, variant, precision):
    print("impermeable", n1, n2, nu, variant, precision, flush=True)
    p = params(N1=n1, N2=n2, nu=nu, avgproc=1, mu_inj=1 / 20., eps=EPS)
    K = np.ones((n1 + 4, n2 + 4))
    a, b = max(4, n1 // 4 // 16 * 16) + 2, max(4, n2 // 4 // 16 * 16) + 2   # from the edge of a coarse cell
    dead = np.zeros(K.shape, bool)
    dead[a:a + max(2, n1 // 3), b:b + max(2, n2 // 3)] = True
    dead[n1 * 3 // 4 + 2, n2 // 4 + 2:n2 * 3 // 4] = True
    K[dead] = 0.
    o, g = pair(p, K, mg_variant=variant, precision=precision)
    g.set_source(o.source())
    g.set_concentration(smooth_c(o))
    its, rr = g.pressure_solve()
    out = o.interior(g.get_pressure()).copy()
    g.close()
    assert rr <= EPS
    return out, ~dead[2:-2, 2:-2], its


@pytest.mark.parametrize("n1,n2,nu,precision", [
    (20, 24, 1.0, 0), (64, 64, 1.0, 0), (130, 130, 1.0, 0), (130, 130, 1.0, 1), (200, 141, 1.0, 0), (260, 260, 1.0, 0),
    (260, 260, 1.0, 2), (130, 130, 2 / 3, 0),
])
def test_zero_permeability_region(gpu_lib, n1, n2, nu, precision):
    x, live, its = _solve(n1, n2, nu, 0, precision)
    y, _, ref = _solve(n1, n2, nu, 1, 0)
    assert np.isfinite(x).all()
    assert np.abs(x - y)[live].max() < 1e-5 * np.abs(y[live]).max(), (its, ref)
