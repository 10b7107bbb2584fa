"""The walk that visits two records a round (a quad's), and one lane's, where
their stacks grow: rods along the three axes, whose inner boxes hold nearly
every point while the leaves hold few, so a walk defers up to 19 entries (the
LDS part of a stack holds 16, a look-ahead starts at five or less).  Against
the binary walk, bit for bit, for points and steps about the largest launch
that takes quads."""
import numpy as np
import pytest

from simulator_amd import _lib as L
from simulator_amd import scene as S
from simulator_amd.simulator import Simulator

from helpers import collider_sim
from test_gpu_build_sizes import still
from test_gpu_quads import sheet

pytestmark = pytest.mark.gpu


def rods(m):
    rng = np.random.default_rng(m)
    c = rng.uniform(-0.9, 0.9, size=(m, 1, 3))
    d = rng.normal(scale=2e-3, size=(m, 3, 3))
    i, ax = np.arange(m), rng.integers(0, 3, m)
    d[i, 0, ax] -= 1
    d[i, 1, ax] += 1
    return (c + d).astype(np.float32).reshape(-1, 3), np.arange(3 * m, dtype=np.uint32).reshape(-1, 3)


@pytest.mark.parametrize("mode", ["static", "rebuild"])
@pytest.mark.parametrize("m,n", [(300, 1), (300, 98304), (300, 98305), (100000, 333)])
def test_deep_stacks(gpu, m, n, mode):
    v, t = rods(m)
    kw = {}
    if mode == "rebuild":
        caps, motion = still(v.shape[0])
        kw = dict(mode=L.CC_BODY_REBUILD, caps=caps, motion=motion)
    a, b = (collider_sim(v, t, depth=1e-3, **kw) for _ in range(2))
    b.set_bvh_width(2)
    for s in (a, b):
        s.simulate(1)
    pts = np.random.default_rng(n).uniform(-1, 1, size=(n, 3)).astype(np.float32)
    got, want = a.collide_points(pts), b.collide_points(pts)
    for x, y in zip(got, want):
        np.testing.assert_array_equal(x, y)
    for s in (a, b):
        s.check_finite()
        s.close()


@pytest.mark.parametrize("n", [98304, 98305])
def test_step_about_the_largest_quad_launch(gpu, n):
    pos, springs = sheet(n, 12, n)
    a, b = (Simulator(pos, springs, S.sphere_body(3), S.params(k=(2.0, 1.0, 0.5), box_depth=0.05)) for _ in range(2))
    b.set_bvh_width(2)
    for s in (a, b):
        s.simulate(3)
    for x, y in zip(a.get_state(), b.get_state()):
        np.testing.assert_array_equal(x, y)
    assert np.any(a.get_state()[2] != 0)
    for s in (a, b):
        s.check_finite()
        s.close()
