"""Bodies whose vertices the caller replaces (cc_body_set_vertices): a static
body is then built and folded on the device.  Against a simulator created over
the new vertices, bit for bit: trees, states through captured blocks recorded
before and after, and queries; at sizes about a chunk of the build, with the
binary walk selected in between, and for a refitted body."""
import numpy as np
import pytest

from simulator_amd import _lib as L
from simulator_amd import scene as S
from simulator_amd.simulator import Simulator

pytestmark = pytest.mark.gpu


def scene(body, side=33):
    return S.grid_scene("posed", side, 1e-3, 0, body, box_depth=0.005, y0=0.95)


def turned(v, a):
    c, s = np.cos(a), np.sin(a)
    P = np.array([0.5, 0.6, 0.0])
    return np.ascontiguousarray((v - P) @ np.array([[c, 0, s], [0, 1, 0], [-s, 0, c]]).T + P, np.float32)


def assert_equal_to_fresh(sim, sc, body, verts, steps):
    fresh = Simulator.from_scene(scene(S.Body(verts, body.tris, body.normals, body.mode, False, body.caps, body.motion),
                                       sc.nx))
    fresh.set_state(*sim.get_state())
    fresh.set_frame(sim.frame)
    a, b = sim.bvh_export(), fresh.bvh_export()
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    rng = np.random.default_rng(1)
    pts = (verts[rng.integers(0, verts.shape[0], 3000)] + rng.normal(scale=3e-3, size=(3000, 3))).astype(np.float32)
    for x, y in zip(sim.collide_points(pts), fresh.collide_points(pts)):
        np.testing.assert_array_equal(x, y)
    for n in steps:
        sim.simulate(n)
        fresh.simulate(n)
        for x, y in zip(sim.get_state(), fresh.get_state()):
            np.testing.assert_array_equal(x, y)
    contacts = int(np.any(sim.get_state()[2] != 0, axis=1).sum())
    fresh.close()
    return contacts


@pytest.mark.parametrize("detail", [(4, 2, 2), (16, 4, 3), (64, 14, 6)])
def test_posed_static_body(gpu, detail):
    body = S.capsules(*detail, L.CC_BODY_STATIC)
    sc = scene(body)
    sim = Simulator.from_scene(sc)
    sim.simulate(2 * sim.block_steps + 1)              # blocks over the body as created
    contacts = 0
    for k in range(3):
        v = turned(body.verts, 0.05 * (k + 1))
        sim.set_body_vertices(v)
        np.testing.assert_array_equal(sim.body_vertices(), v)
        assert sim.bvh_width()[0] == 4
        if k == 1:                                     # the binary walk, and back
            sim.set_bvh_width(2)
            sim.simulate(1)
            sim.set_bvh_width(4)
        contacts += assert_equal_to_fresh(sim, sc, body, v, (1, sim.block_steps, 2))
    sim.bvh_rebuild()
    assert_equal_to_fresh(sim, sc, body, v, (1,))
    assert contacts > 0
    sim.close()


def test_posed_single_and_two_triangles(gpu):
    v = np.float32([[0, 0, 0], [1, 0, 0], [0, 0, 1], [1, 0, 1]])
    for t in ([[0, 2, 1]], [[0, 2, 1], [1, 2, 3]]):
        body = S.Body(v, np.uint32(t), np.zeros_like(v), L.CC_BODY_STATIC, False)
        sc = scene(body, 9)
        sim = Simulator.from_scene(sc)
        up = v + np.float32([0, 0.9, 0])
        sim.set_body_vertices(up)
        sim.simulate(40)
        fresh = Simulator.from_scene(scene(S.Body(up, np.uint32(t), np.zeros_like(v), L.CC_BODY_STATIC, False), 9))
        fresh.simulate(40)
        for x, y in zip(sim.get_state(), fresh.get_state()):
            np.testing.assert_array_equal(x, y)
        sim.close()
        fresh.close()


def test_posed_refitted_body(gpu):
    body = S.capsules(16, 4, 3, L.CC_BODY_REFIT)
    sc = scene(body)
    sim = Simulator.from_scene(sc)
    sim.simulate(2 * sim.block_steps)
    v = np.ascontiguousarray(body.verts * np.float32([1.0, 1.0, 0.7]))   # another topology
    sim.set_body_vertices(v)
    x0 = sim.get_state()
    other = Simulator.from_scene(sc)
    other.set_frame(sim.frame)
    other.set_body_vertices(v)
    other.set_state(*x0)
    for n in (sim.block_steps, 3, sim.block_steps):
        sim.simulate(n)
        other.simulate(n)
        for x, y in zip(sim.get_state(), other.get_state()):
            np.testing.assert_array_equal(x, y)
    sim.close()
    other.close()
