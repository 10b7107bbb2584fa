"""The LBVH build at the sizes where its parts change: sort tiles of 1,024
keys and the 64 tiles up to which a scatter sums the tiles' counts itself, and
the tree's chunks of 1,024 leaves, eight of them to a workgroup of the next
level.  Keys, order, links and boxes against the oracle bit for bit, for a
static body (searches and refit) and a rebuilt one (by splits), over spread
triangles and over many of one Morton code."""
import numpy as np
import pytest

from simulator_amd import _lib as L

from helpers import assert_bvh_equal, collider_sim, oracle_bvh

pytestmark = pytest.mark.gpu


def soup(m, kind, seed):
    """m small triangles; "clumped": all centres in a few cells, so that runs
    of equal codes are split by their primitives alone."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(-1, 1, size=(m, 1, 3))
    if kind == "clumped":
        c = np.round(c * 1.5) / 1.5
    v = (c + rng.normal(scale=1e-3, size=(m, 3, 3))).astype(np.float32).reshape(-1, 3)
    return v, np.arange(3 * m, dtype=np.uint32).reshape(-1, 3)


def still(nv):
    """One capsule over all vertices and no motion."""
    caps = {"vstart": np.array([0, nv], np.uint32), "p0": np.zeros((1, 3), np.float32),
            "p1": np.float32([[0, 1, 0]]), "radius": np.ones(1, np.float32), "phase": np.zeros(1, np.float32)}
    return caps, dict(amp=0.0, freq=0.0, rot_amp=0.0, breath_amp=0.0, breath_freq=0.0, dir=(1, 0, 0),
                      pivot=(0, 0, 0))


@pytest.mark.parametrize("kind", ["spread", "clumped"])
@pytest.mark.parametrize("m", [1, 2, 3, 1023, 1024, 1025, 2048, 8191, 8193, 9217, 65536, 65537])
def test_build_sizes(gpu, m, kind):
    v, t = soup(m, kind, m)
    sim = collider_sim(v, t)
    assert_bvh_equal(sim.bvh_export(), oracle_bvh(v, t, 0.01))
    sim.close()
    caps, motion = still(v.shape[0])
    sim = collider_sim(v, t, mode=L.CC_BODY_REBUILD, caps=caps, motion=motion)
    sim.simulate(1)
    pose = sim.body_vertices()
    assert_bvh_equal(sim.bvh_export(), oracle_bvh(pose, t, 0.01))
    sim.close()
