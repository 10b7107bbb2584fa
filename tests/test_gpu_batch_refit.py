"""Refitted bodies of a batch, by levels over tables of all of them, beside
static, rebuilt and missing bodies: sizes about the group of 1,024 leaves, one
and two triangles, alone and together.  Poses and trees of every instance
against its own simulator, bit for bit, in single launches and graph blocks."""
import numpy as np
import pytest

from simulator_amd import _lib as L
from simulator_amd import batch as B
from simulator_amd import scene as S
from simulator_amd.simulator import Simulator

from test_gpu_build_sizes import soup
from test_gpu_refit_levels import moving

pytestmark = pytest.mark.gpu


def instance(k, m, mode):
    sc = S.grid_scene("r", 8 + k, 1e-3, 0, None, box_depth=0.01, seed=k, y0=0.95)
    if mode != L.CC_BODY_NONE:
        v, t = soup(m, "spread" if k % 2 else "clumped", m + k)
        caps, motion = moving(v.shape[0])
        sc.body = S.Body(v, t, np.zeros_like(v), mode, False, caps, motion)
    return sc


RF, RB, ST, NO = L.CC_BODY_REFIT, L.CC_BODY_REBUILD, L.CC_BODY_STATIC, L.CC_BODY_NONE


@pytest.mark.parametrize("bodies", [
    [(1, RF)], [(2, RF)], [(1025, RF)],
    [(3, RF), (1024, RF), (1025, RF), (2, RF), (9217, RF), (1, RF)],
    [(700, ST), (1500, RF), (0, NO), (2100, RB), (1, RF), (1023, RF), (5, RB)]])
def test_batch_refit(gpu, bodies):
    scs = [instance(k, m, mode) for k, (m, mode) in enumerate(bodies)]
    b = B.Batch(scs)
    sims = [Simulator.from_scene(sc) for sc in scs]
    for steps in (1, 16, 3):
        b.simulate(steps)
        for s in sims:
            s.simulate(steps)
        for k, s in enumerate(sims):
            for g, w in zip(b.get_state(k), s.get_state()):
                np.testing.assert_array_equal(g, w, err_msg=f"instance {k}")
            if bodies[k][1] == NO:
                continue
            verts, tree = b.body_export(k)
            np.testing.assert_array_equal(verts, s.body_vertices())
            want = s.bvh_export()
            for key in want:
                np.testing.assert_array_equal(tree[key], want[key], err_msg=f"instance {k}: {key}")
    b.close()
    for s in sims:
        s.close()
