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
