"""The step and the point query with four lanes per vertex (k_verlet_quad,
k_collide_quad) against one lane per vertex walking the binary tree, bit for
bit: cloth sizes about the edges of a wave's 16 quads and a workgroup's 64,
rows of at most 12, at most 24 and more springs, empty rows and pins, and
point counts about the largest that takes quads."""
import numpy as np
import pytest

from simulator_amd import _lib as L
from simulator_amd import scene as S
from simulator_amd.simulator import Simulator

pytestmark = pytest.mark.gpu


def sheet(n, degree, seed):
    """n vertices about the sphere's surface, up to `degree` springs each (a
    few rows empty), three types."""
    rng = np.random.default_rng(seed)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    pos = (np.array([0.5, 0.5, 0.0]) + d * rng.uniform(0.295, 0.306, size=(n, 1))).astype(np.float32)
    sets = []
    for t in range(3):
        most = degree // 3
        k = rng.integers(0, most + 1, size=n)
        k[rng.random(n) < 0.1] = 0
        k[0] = most                                   # the widest row is there
        row = np.zeros(n + 1, np.uint32)
        np.cumsum(k, out=row[1:])
        end = rng.integers(0, n, size=int(row[-1]))
        src = np.repeat(np.arange(n), k)
        end = np.where(end == src, (end + 1) % n, end)
        col = np.zeros(int(row[-1]), L.SPRING_DTYPE)
        col["end"] = end
        col["original"] = np.linalg.norm(pos[src] - pos[end], axis=1)
        sets.append((row, col))
    return pos, sets


@pytest.mark.parametrize("mode", ["static", "rebuild"])
@pytest.mark.parametrize("degree", [12, 24, 27])
@pytest.mark.parametrize("n", [2, 15, 16, 17, 63, 64, 65, 300])
def test_quad_step_equals_one_lane(gpu, n, degree, mode):
    pos, springs = sheet(n, degree, 100 * n + degree)
    if mode == "static":
        body = S.sphere_body(3)
    else:                                             # split records
        body = S.capsules(16, 4, 3, L.CC_BODY_REBUILD)
        pos += np.float32([0.0, 0.1, 0.0])
    prm = S.params(k=(2.0, 1.0, 0.5), box_depth=0.05)
    pins = np.arange(0, n, 9, dtype=np.uint32) if n > 9 else None
    a, b = (Simulator(pos, springs, body, prm, pins) for _ in range(2))
    b.set_bvh_width(2)
    assert a.bvh_width()[0] == 4 and b.bvh_width()[0] == 2
    contacts = 0
    for steps in (1, 1, a.block_steps, 3):
        a.simulate(steps)
        b.simulate(steps)
        for x, y in zip(a.get_state(), b.get_state()):
            np.testing.assert_array_equal(x, y)
        contacts += int(np.any(a.get_state()[2] != 0, axis=1).sum())
    assert contacts > 0 or n < 15 or mode == "rebuild"
    a.close()
    b.close()


@pytest.mark.parametrize("n", [1, 63, 65, 65535, 65536, 65537])
def test_quad_query_equals_one_lane(gpu, n):
    rng = np.random.default_rng(n)
    d = rng.normal(size=(n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    pts = (np.array([0.5, 0.5, 0.0]) + d * rng.uniform(0.28, 0.32, size=(n, 1))).astype(np.float32)
    a, b = (Simulator.from_scene(S.small(side=8)) for _ in range(2))
    b.set_bvh_width(2)
    for x, y in zip(a.collide_points(pts), b.collide_points(pts)):
        np.testing.assert_array_equal(x, y)
    a.close()
    b.close()
