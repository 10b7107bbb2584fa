"""A box depth changed on a live simulator (cc_sim_set_params, cc_sim_load)
takes effect for the body of every mode.  A refitted body's trees and states
against the chunked refit's (CC_REBUILD_BOTTOM_UP=0, the same topology), bit
for bit, and every body's leaf boxes against those of a simulator created with
the depth (its tree has another order: matched by primitive), in the four-wide
and in the binary form."""
import numpy as np
import pytest

from simulator_amd import _lib as L
from simulator_amd import scene as S
from simulator_amd.simulator import Simulator

pytestmark = pytest.mark.gpu

MODES = [L.CC_BODY_STATIC, L.CC_BODY_REFIT, L.CC_BODY_REBUILD]
DEEP = 0.03


def scene(mode, depth=0.002):
    return S.grid_scene("depth", 33, 1e-3, 0, S.capsules(16, 4, 3, mode), box_depth=depth, y0=0.93)


def deepen(sim, how, tmp_path):
    if how == "set":
        p = sim.params
        p.box_depth = DEEP
        sim.set_params(p)
        return
    path = str(tmp_path / "deep.ckpt")
    other = Simulator.from_scene(scene(L.CC_BODY_STATIC, DEEP))
    other.set_state(*sim.get_state())
    other.set_frame(sim.frame)
    other.save(path)
    other.close()
    sim.load(path)


def leaf_boxes(sim):
    t = sim.bvh_export()
    out = np.empty_like(t["box_leaf"])
    out[t["order"]] = t["box_leaf"]
    return out


@pytest.mark.parametrize("how", ["set", "load"])
@pytest.mark.parametrize("width", [4, 2])
@pytest.mark.parametrize("mode", MODES)
def test_leaf_boxes_follow_the_depth(gpu, mode, width, how, tmp_path):
    sim, deep = Simulator.from_scene(scene(mode)), Simulator.from_scene(scene(mode, DEEP))
    for s in (sim, deep):
        s.set_bvh_width(width)
        s.simulate(5)
    deepen(sim, how, tmp_path)
    for steps in (0, 1, 4):
        for s in (sim, deep):
            s.simulate(steps)
        np.testing.assert_array_equal(sim.body_vertices(), deep.body_vertices())
        np.testing.assert_array_equal(leaf_boxes(sim), leaf_boxes(deep), err_msg=f"after {steps} steps")
    sim.close()
    deep.close()


@pytest.mark.parametrize("how", ["set", "load"])
@pytest.mark.parametrize("width", [4, 2])
def test_levels_equal_chunks_at_the_new_depth(gpu, width, how, tmp_path, monkeypatch):
    sims = []
    for up in ("1", "0"):
        monkeypatch.setenv("CC_REBUILD_BOTTOM_UP", up)
        sims.append(Simulator.from_scene(scene(L.CC_BODY_REFIT)))
    contacts = 0
    for s in sims:
        s.set_bvh_width(width)
        s.simulate(150)
        deepen(s, how, tmp_path)
    for steps in (1, sims[0].block_steps, 3):
        for s in sims:
            s.simulate(steps)
        for x, y in zip(*(s.get_state() for s in sims)):
            np.testing.assert_array_equal(x, y)
        a, b = (s.bvh_export() for s in sims)
        for k in a:
            np.testing.assert_array_equal(a[k], b[k], err_msg=k)
        contacts += int(np.any(sims[0].get_state()[2] != 0, axis=1).sum())
    assert contacts > 0
    for s in sims:
        s.close()
