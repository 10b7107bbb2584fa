"""States, points and body vertices between host arrays and the device, in
chunks of 65,536 through pinned memory that a handle keeps: sizes about one and
two chunks, calls that grow and shrink, partial reads, and several threads on
one handle.  Exact."""
import threading

import numpy as np
import pytest

from simulator_amd import _lib as L
from simulator_amd import scene as S
from simulator_amd.simulator import Simulator

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 65535, 65537, 131072, 131073, 200001])
def test_state_read_back(gpu, n):
    rng = np.random.default_rng(n)
    want = [rng.normal(size=(n, 3)).astype(np.float32) for _ in range(3)]
    sim = Simulator(want[0], [(np.zeros(n + 1, np.uint32), np.zeros(0, L.SPRING_DTYPE))], None, S.params())
    sim.set_state(*want)
    for x, y in zip(sim.get_state(), want):
        np.testing.assert_array_equal(x, y)
    only = np.zeros((n, 3), np.float32)                     # the other two arrays NULL
    L.check(L.lib().cc_sim_get_state(sim._h, None, L.ptr(only), None))
    np.testing.assert_array_equal(only, want[1])
    sim.close()


def test_queries_grow_and_shrink(gpu):
    sim = Simulator.from_scene(S.small(side=8))
    rng = np.random.default_rng(0)
    d = rng.normal(size=(131073, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    pts = (np.array([0.5, 0.5, 0.0]) + d * rng.uniform(0.28, 0.32, size=(d.shape[0], 1))).astype(np.float32)
    whole = sim.collide_points(pts)
    for k in (0, 1, 1000, 65536, 65537, 131072):
        for x, y in zip(sim.collide_points(pts[:k]), whole):
            np.testing.assert_array_equal(x, y[:k])
    assert whole[1].any() and not whole[1].all()

    out, per = {}, 20000

    def query(t):
        out[t] = [sim.collide_points(pts[t * per:(t + 1) * per]) for _ in range(5)]

    threads = [threading.Thread(target=query, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for t in range(4):
        for got in out[t]:
            for x, y in zip(got, whole):
                np.testing.assert_array_equal(x, y[t * per:(t + 1) * per])
    sim.close()


@pytest.mark.parametrize("nv", [3, 65536, 65538, 196611])
def test_body_vertices(gpu, nv):
    rng = np.random.default_rng(nv)
    v = rng.uniform(-1, 1, size=(nv, 3)).astype(np.float32)
    m = min(nv // 3, 3000)
    tris = np.arange(3 * m, dtype=np.uint32).reshape(-1, 3)
    body = S.Body(v, tris, np.zeros_like(v), L.CC_BODY_STATIC, False, None, {})
    sim = Simulator(np.zeros((1, 3), np.float32), [(np.zeros(2, np.uint32), np.zeros(0, L.SPRING_DTYPE))], body,
                    S.params(box_depth=0.01))
    for _ in range(3):
        v = rng.uniform(-1, 1, size=(nv, 3)).astype(np.float32)
        sim.set_body_vertices(v)
        np.testing.assert_array_equal(sim.body_vertices(), v)
    sim.close()
