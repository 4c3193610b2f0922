"""The 5-point V-cycle's tile legs and bottom (2 x 2 blocks in LDS) against the
one-kernel-per-pass cycle (mg_variant 1), which does the same operations in the
same colour order on faces formed by division: stopped after three CG iterations
both must hold the same iterate.  The faces differ by the rounding of a reciprocal
(about 2^-52) and sums by theirs; three cycles amplify that by at most ten times
the condition number, about 2060^2 at the largest size: 1e-8, doubled.  The FP32
cycle rounds about a hundred operations per cell and cycle at 2^-24: with the same
ten over three iterations 2e-4.  A halo one block too narrow leaves out the last
dependence of the cells at the tiles' edges, about 4^-4 of the local correction; a
tile at a wrong origin leaves cells unsmoothed.
Sizes: sides of one octave (the coarsest level is 2 x 2: on a level one cell wide
mg_variant 1 keeps couplings across the boundary), whose first coarse level is the
bottom's (up to 128), just above it, around one and two tiles' writes, clamped last
tiles, ragged, oblong, several tile levels, and above the tiles' limit of 1024."""
import numpy as np
import pytest

from helpers import pair, params, rel_err, smooth_c

pytestmark = pytest.mark.gpu

SIZES = [(5, 8), (20, 31), (33, 64), (100, 127), (128, 128), (129, 130), (130, 250), (208, 210), (234, 209), (256, 256),
         (257, 258), (260, 511), (417, 300), (700, 1001), (1030, 2048), (2049, 2060)]


def _iterate(n1, n2, avg, sweeps, precision, variant):
    from impec2d_amd import capi
    print("blocks5", n1, n2, avg, sweeps, precision, variant, flush=True)
    p = params(N1=n1, N2=n2, nu=1.0, avgproc=avg, mu_inj=1 / 20., eps=1e-13, max_iter=3)
    K = np.exp(0.5 * np.random.default_rng(n1 * 1000 + n2).standard_normal((n1 + 4, n2 + 4)))
    o, g = pair(p, K, mg_variant=variant, mg_pre=sweeps, mg_post=sweeps, precision=precision)
    g.set_source(o.source())
    g.set_concentration(smooth_c(o))
    with pytest.raises(capi.ImpecError) as e:
        g.pressure_solve()
    assert e.value.code == capi.IMPEC_ENOCONV
    out = o.interior(g.get_pressure()).copy()
    g.close()
    assert np.isfinite(out).all()
    return out


@pytest.mark.parametrize("avg,sweeps,precision", [(0, 2, 0), (1, 1, 0), (0, 1, 1), (1, 2, 1)])
@pytest.mark.parametrize("n1,n2", SIZES)
def test_tile_cycle_equals_unfused_cycle(gpu_lib, n1, n2, avg, sweeps, precision):
    x = _iterate(n1, n2, avg, sweeps, precision, 0)
    y = _iterate(n1, n2, avg, sweeps, 0, 1)
    assert rel_err(x, y) < (2e-4 if precision else 2e-8)
