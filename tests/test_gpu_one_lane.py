"""The step with one lane per vertex through the four-wide form, beyond the
largest cloth that takes four (read from the source, so that another limit
cannot empty these tests): walks whose stacks grow past the 16 entries held in
LDS (with four lanes too), over a static and a rebuilt body, bit for bit
against the binary walk."""
import os
import re

import numpy as np
import pytest

import oracle as O
from simulator_amd import _lib as L
from simulator_amd import scene as S
from simulator_amd.simulator import Simulator

from test_gpu_build_sizes import still
from test_gpu_quads import sheet
from test_grouped_walk_model import fold, walk

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def quad_max_n():
    with open(os.path.join(ROOT, "simulator_amd", "csrc", "cc_sim.h")) as f:
        return int(re.search(r"constexpr uint32_t QUAD_MAX_N = (\d+);", f.read()).group(1))


def flat(c, h, axis):
    """A triangle whose box is c +- h but for `axis`, where it is flat."""
    u, w = [a for a in range(3) if a != axis]
    v = np.tile(np.asarray(c, float), (3, 1))
    v[0, u] -= h
    v[1, u] += h
    v[:2, w] -= h
    v[2, w] += h
    return v


def chain():
    """A body whose tree is a chain of 24 nodes: the centres of group k lie in
    the cell of Morton code bit k beside a common cell (cells of edge 1), so
    every group of four splits off alone.  A group's pairs cross (flat in y and
    flat in x): the boxes of its three nodes hold every point about the middle
    and those of its triangles hold none, so the walk defers a node at every
    level before it comes to the one triangle whose box holds the point."""
    tris = []
    for bit in range(24):
        c = np.full(3, 256.5)
        c[2 - bit % 3] += 1 << (bit // 3)
        tris += [flat(c, 256.5, 1), flat(c, 256.5, 0)] * 2
    tris += [flat(np.full(3, 512.5), 100.0, 1),                                       # with the larger one below,
             np.array([[300.0, 300, 300], [725, 300, 500], [500, 725, 725]])]         # popped last
    tris.append(np.full((3, 3), 1023.0) + np.eye(3))                                  # the far corner of the root box
    v = np.concatenate(tris).astype(np.float32)
    return v, np.arange(v.shape[0], dtype=np.uint32).reshape(-1, 3)


def points(n):
    return np.random.default_rng(n).uniform(390, 510, size=(n, 3)).astype(np.float32)


def test_the_chain_defers_more_than_lds_holds():
    v, t = chain()
    recs = fold(O.bvh_build(v, t, 1e-3))
    r = [walk(recs, p) for p in points(50)]
    assert max(most for _, _, most in r) > 16 + 3, r
    assert all(hit >= 0 for hit, _, _ in r), r


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["static", "rebuild"])
@pytest.mark.parametrize("n", [300, quad_max_n() + 1])            # four lanes, one lane
def test_deep_stacks(gpu, n, mode):
    v, t = chain()
    caps, motion = still(v.shape[0]) if mode == "rebuild" else (None, {})
    body = S.Body(v, t, np.zeros_like(v), L.CC_BODY_REBUILD if mode == "rebuild" else L.CC_BODY_STATIC, False, caps,
                  motion)
    none = [(np.zeros(n + 1, np.uint32), np.zeros(0, L.SPRING_DTYPE))]
    a, b = (Simulator(points(n), none, body, S.params(box_depth=1e-3)) for _ in range(2))
    b.set_bvh_width(2)
    assert a.bvh_width()[0] == 4 and b.bvh_width()[0] == 2
    for s in (a, b):
        s.set_debug(True)
    contacts = 0
    for steps in (1, 1, a.block_steps + 1):
        for s in (a, b):
            s.simulate(steps)
            s.check_finite()
        for x, y in zip(a.get_debug(), b.get_debug()):
            np.testing.assert_array_equal(x, y)
        for x, y in zip(a.get_state(), b.get_state()):
            np.testing.assert_array_equal(x, y)
        contacts += int(np.any(a.get_state()[2] != 0, axis=1).sum())
    assert contacts > n / 100, contacts
    a.close()
    b.close()


@pytest.mark.gpu
@pytest.mark.parametrize("degree", [12, 24, 27])
def test_rows_with_one_lane(gpu, degree):
    pos, springs = sheet(quad_max_n() + 1, degree, degree)
    pos += np.float32([0.0, 0.1, 0.0])
    body = S.capsules(16, 4, 3, L.CC_BODY_REBUILD)
    a, b = (Simulator(pos, springs, body, S.params(k=(2.0, 1.0, 0.5), box_depth=0.05)) for _ in range(2))
    b.set_bvh_width(2)
    for s in (a, b):
        s.simulate(3)
        s.check_finite()
    for x, y in zip(a.get_state(), b.get_state()):
        np.testing.assert_array_equal(x, y)
    assert np.any(a.get_state()[2] != 0)
    a.close()
    b.close()
