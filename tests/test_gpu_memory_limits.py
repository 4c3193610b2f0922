"""What happens at the end of memory.  A child process loads tests/host/alloc_limit.c
before the library, so that allocations fail where the test wants them to: fields
are read without pinned staging memory, many readers at a time neither fail nor
allocate staging memory again and again, and the planes of the 9-point cycle, which
a solve can do without, never take the room of what a context needs."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HEAD = """
import ctypes, sys, threading
import numpy as np
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
shim.alloc_limit.argtypes = [ctypes.c_size_t, ctypes.c_size_t]
shim.alloc_live.restype = ctypes.c_size_t
ANY = 2 ** 64 - 1
from impec2d_amd import capi

def fields(n1, n2, seed):
    g = capi.Context(capi.default_params(N1=n1, N2=n2))
    rng = np.random.default_rng(seed)
    c, p, v = (rng.standard_normal(s) for s in (g.scalar_shape(), g.scalar_shape(), g.velocity_shape()))
    g.set_concentration(c)
    g.set_pressure(p)
    g.set_velocity(v)
    return g, c, p, v

def check(g, c, p, v):
    assert np.array_equal(g.get_concentration(), c)
    assert np.array_equal(g.get_pressure(), p)
    assert np.array_equal(g.get_velocity(), v)
"""


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("shim") / "alloc_limit.so")
    src = os.path.join(ROOT, "tests", "host", "alloc_limit.c")
    subprocess.check_call(["gcc", "-shared", "-fPIC", "-O1", "-Wall", src, "-o", so, "-ldl", "-lpthread"])
    return so


def _child(shim, body):
    r = subprocess.run([sys.executable, "-c", HEAD + body, shim], cwd=ROOT, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, timeout=100, text=True)
    assert r.returncode == 0 and "done" in r.stdout, r.stdout


def test_fields_are_read_without_pinned_memory(gpu_lib, shim):
    _child(shim, """
for n1, n2 in ((2, 2), (65, 63), (723, 721), (1021, 1025)):
    shim.alloc_limit(ANY, 1 << 20)
    g, c, p, v = fields(n1, n2, n1)
    check(g, c, p, v)
    shim.alloc_limit(ANY, ANY)   # memory again
    check(g, c, p, v)
    g.close()
print("done")
""")


def test_many_readers_share_a_bounded_number_of_stages(gpu_lib, shim):
    """Twelve threads with contexts of their own read eight times each; the staging
    memory stays allocated while contexts exist, at most eight pieces of it, and what
    finds none free is read without."""
    _child(shim, """
state = [fields(700 + 31 * k, 600 + 17 * k, k) for k in range(12)]
failed = []
def work(s):
    try:
        for _ in range(8):
            check(*s)
    except BaseException as e:
        failed.append(repr(e))
threads = [threading.Thread(target=work, args=(s,)) for s in state]
for t in threads: t.start()
for t in threads: t.join()
assert not failed, failed
assert 1 <= shim.alloc_host_calls() <= 8, shim.alloc_host_calls()
print("done")
""")


def test_planes_of_the_nine_point_cycle_make_room(gpu_lib, shim):
    """Limits one byte short of everything, of everything but the permeability, and of
    half the planes: a context is created and solves wherever one without planes
    (mg_variant 1) fits, and has them only where they fit beside the rest."""
    _child(shim, """
n1, n2, eps = 96, 130, 1e-9
q = np.zeros((n1, n2))
q[0, 0], q[-1, -1] = n1 * n2, -n1 * n2
K = [np.exp(0.3 * np.random.default_rng(s).standard_normal((n1 + 4, n2 + 4))) for s in (1, 2)]

def run(variant, limit, late):
    shim.alloc_limit(limit, ANY)
    g = capi.Context(capi.default_params(N1=n1, N2=n2, nu=2 / 3, eps=eps, diffusion=1, mg_variant=variant))
    created = shim.alloc_live()
    g.set_source(q)
    if late:
        g.set_permeability(*K)
    its, rr = g.pressure_solve()
    assert rr <= eps
    p, live = g.get_pressure(), shim.alloc_live()
    g.close()
    assert shim.alloc_live() == 0
    return p, created, live

plain, need0, _ = run(1, ANY, False)
plain_late, _, need = run(1, ANY, True)
full, all0, _ = run(0, ANY, False)
full_late, _, everything = run(0, ANY, True)
planes = all0 - need0
assert planes > 100 * n1 * n2 and everything - need == planes
top = np.abs(plain).max(), np.abs(plain_late).max()
for limit, late in ((everything - 1, False), (everything - 1, True), (need + planes // 2, True), (need, True),
                    (all0, False)):
    p, created, live = run(0, limit, late)
    assert created in (need0, all0) and live <= limit
    assert created == (all0 if limit >= all0 else need0), (created, limit)
    want = plain_late if late else plain
    assert np.abs(p - want)[2:-2, 2:-2].max() < 1e-4 * top[late], limit
print("done")
""")
