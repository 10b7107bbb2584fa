"""Refits by levels against refits by chunks (CC_REBUILD_BOTTOM_UP=0), bit for
bit: trees and states of a deforming refitted body, in the four-wide and in the
binary form, at sizes about the group of 1,024 leaves and where the levels
grow to three; over spread triangles and over many of one Morton code."""
import numpy as np
import pytest

from simulator_amd import _lib as L

from helpers import collider_sim
from test_gpu_build_sizes import soup

pytestmark = pytest.mark.gpu


def moving(nv):
    """Two capsules, one per half of the vertices, that swing and breathe."""
    caps = {"vstart": np.array([0, nv // 2, nv], np.uint32), "p0": np.zeros((2, 3), np.float32),
            "p1": np.float32([[0, 1, 0], [1, 0, 0]]), "radius": np.ones(2, np.float32),
            "phase": np.float32([0.0, 0.7])}
    return caps, dict(amp=0.1, freq=3.0, rot_amp=0.3, breath_amp=0.05, breath_freq=2.0, dir=(1, 0, 0),
                      pivot=(0, 0.5, 0))


@pytest.mark.parametrize("kind", ["spread", "clumped"])
@pytest.mark.parametrize("m", [2, 3, 1023, 1024, 1025, 2049, 9217, 70001])
def test_refit_levels(gpu, m, kind, monkeypatch):
    v, t = soup(m, kind, m)
    caps, motion = moving(v.shape[0])
    sims = []
    for up in ("1", "0"):
        monkeypatch.setenv("CC_REBUILD_BOTTOM_UP", up)
        sims.append(collider_sim(v, t, mode=L.CC_BODY_REFIT, caps=caps, motion=motion))
    for width in (4, 2, 4):
        for s in sims:
            s.set_bvh_width(width)
        for steps in (1, 6):
            for s in sims:
                s.simulate(steps)
            a, b = (s.bvh_export() for s in sims)
            for k in a:
                np.testing.assert_array_equal(a[k], b[k], err_msg=f"{k} width {width} steps {steps}")
        pts = (sims[0].body_vertices()[:3000] + np.float32(1e-3)).astype(np.float32)
        for x, y in zip(*(s.collide_points(pts) for s in sims)):
            np.testing.assert_array_equal(x, y)
    for s in sims:
        s.close()
