"""Fields read back in chunks through staging memory: what was set comes back bit
for bit, whatever the sizes (one chunk, a ragged last chunk, an odd row pitch,
more than one staging half, several copying threads), also from several threads
and contexts at a time.  Copies only: exact equality."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ctx(n1, n2):
    from impec2d_amd import capi
    return capi.Context(capi.default_params(N1=n1, N2=n2))


def _round_trip(n1, n2, seed):
    g = _ctx(n1, n2)
    rng = np.random.default_rng(seed)
    c, p, v = rng.standard_normal(g.scalar_shape()), rng.standard_normal(g.scalar_shape()), \
        rng.standard_normal(g.velocity_shape())
    g.set_concentration(c)
    g.set_pressure(p)
    g.set_velocity(v)
    for _ in range(2):
        assert np.array_equal(g.get_concentration(), c)
        assert np.array_equal(g.get_velocity(), v)
        assert np.array_equal(g.get_pressure(), p)
    g.close()


@pytest.mark.parametrize("n1,n2", [(2, 2), (3, 200), (65, 63), (723, 721), (1021, 1025), (1537, 1530), (2, 70001)])
def test_fields_come_back_bitwise(gpu_lib, n1, n2):
    _round_trip(n1, n2, n1 + n2)


def test_reads_from_several_threads(gpu_lib):
    failed = []

    def work(k):
        try:
            for q in range(3):
                _round_trip(700 + 31 * k, 600 + 17 * k + q, k)
        except BaseException as e:   # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed[0]


def test_reads_of_one_context_from_several_threads(gpu_lib):
    """A read leaves the context as it is: readers of the same one do not disturb
    each other."""
    g = _ctx(723, 721)
    rng = np.random.default_rng(7)
    c, p, v = rng.standard_normal(g.scalar_shape()), rng.standard_normal(g.scalar_shape()), \
        rng.standard_normal(g.velocity_shape())
    g.set_concentration(c)
    g.set_pressure(p)
    g.set_velocity(v)
    failed = []

    def work(k):
        try:
            for q in range(8):
                get, want = ((g.get_concentration, c), (g.get_velocity, v), (g.get_pressure, p))[(k + q) % 3]
                assert np.array_equal(get(), want)
        except BaseException as e:   # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    g.close()
    assert not failed, failed[0]


@pytest.mark.parametrize("splitting", ["strang", "parallel", "x_first"])
def test_reads_between_steps_change_nothing(gpu_lib, splitting):
    from impec2d_amd import capi
    split = {"strang": capi.SPLIT_STRANG, "parallel": capi.SPLIT_PARALLEL, "x_first": capi.SPLIT_X_FIRST}[splitting]
    end = []
    for reads in (False, True):
        g = capi.Context(capi.default_params(N1=70, N2=91, nu=1.0, mu_res=1.0, mu_inj=0.1, eps=1e-10, para_eps=1e-10,
                                             dim_splitting=split, diffusion=1, alpha_absolute=1, alpha_l=1e-3,
                                             alpha_t=1e-4, d_m=1e-5))
        q = np.zeros((70, 91))
        q[0, 0], q[-1, -1] = 70 * 91, -70 * 91
        g.set_source(q)
        t = 0.0
        for _ in range(5):
            t += g.step(t)
            if reads:
                g.get_concentration(), g.get_velocity(), g.get_pressure()
        end.append((g.get_concentration(), g.get_pressure(), g.get_velocity()))
        g.close()
    assert end[0][0].max() > 0.1
    for a, b in zip(*end):
        assert np.array_equal(a, b)
