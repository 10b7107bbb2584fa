"""The batch's tables: instances dealt to XCDs (many alike) and not (one far
larger than the rest), and a body of more sort tiles than a scatter sums by
itself.  Every instance against its own simulator, bit for bit, states and
body trees, in single launches and in graph blocks."""
import numpy as np
import pytest

from simulator_amd import _lib as L
from simulator_amd import batch as B
from simulator_amd import scene as S
from simulator_amd.simulator import Simulator

pytestmark = pytest.mark.gpu


def instance(side, seg, k, mode):
    v, t, nrm, caps = S.capsule_body(3, 0.1, 0.2, *S.CAPSULE_BOX, seg, max(2, seg // 4), max(2, seg // 4), 50 + k)
    body = S.Body(v, t, nrm, mode, True, caps, S._motion(50 + k))
    return S.grid_scene("b", side, 1e-3, 0, body, box_depth=0.01, seed=k, y0=0.95)


@pytest.mark.parametrize("kind", ["alike", "uneven", "big body"])
def test_batch_tables(gpu, kind):
    if kind == "alike":                   # 8 a XCD
        scs = [instance(17 + k % 3, 12, k, L.CC_BODY_REBUILD) for k in range(64)]
    elif kind == "uneven":
        scs = [instance(40, 40, 0, L.CC_BODY_REBUILD)] + [instance(9, 8, k, L.CC_BODY_REBUILD) for k in range(1, 5)]
    else:                                 # 71,280 triangles: 70 tiles of the sort
        scs = [instance(33, 132, 0, L.CC_BODY_REBUILD), instance(20, 12, 1, L.CC_BODY_REBUILD),
               instance(20, 12, 2, L.CC_BODY_REFIT)]
        assert scs[0].body.tris.shape[0] > 65536
    b = B.Batch(scs)
    sims = [Simulator.from_scene(sc) for sc in scs]
    for steps in (1, 16, 3):
        b.simulate(steps)
        for s in sims:
            s.simulate(steps)
    for k, s in enumerate(sims):
        for g, w in zip(b.get_state(k), s.get_state()):
            np.testing.assert_array_equal(g, w, err_msg=f"instance {k}")
        if kind != "alike" or k % 16 == 0:
            verts, tree = b.body_export(k)
            np.testing.assert_array_equal(verts, s.body_vertices())
            want = s.bvh_export()
            for key in want:
                np.testing.assert_array_equal(tree[key], want[key], err_msg=f"instance {k}: {key}")
        s.close()
    b.close()
