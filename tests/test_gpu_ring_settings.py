"""Settings of a moving body's pipeline that leave little room in its ring of
poses (two per step of a block): a chain of launches takes a frame less where
the default four do not fit beside the lookahead, and only what does not fit
then is refused.  Results are the default settings'."""
import numpy as np
import pytest

from simulator_amd import _lib as L
from simulator_amd import scene as S
from simulator_amd.simulator import Simulator

pytestmark = pytest.mark.gpu

RF, RB = L.CC_BODY_REFIT, L.CC_BODY_REBUILD


def scene(mode):
    return S.grid_scene("ring", 24, 1e-3, 0, S.capsules(16, 4, 3, mode), box_depth=0.01, y0=0.93)


@pytest.mark.parametrize("mode,env", [
    (RB, {"GRAPH_STEPS": 12}), (RF, {"GRAPH_STEPS": 16}),
    (RB, {"GRAPH_STEPS": 16, "BODY_LANES": 3}), (RF, {"GRAPH_STEPS": 16, "BODY_LANES": 3}),
    (RB, {"GRAPH_STEPS": 20, "BODY_LANES": 4}), (RF, {"GRAPH_STEPS": 20, "BODY_LANES": 4}),
    (RB, {"LOOKAHEAD": 33}), (RF, {"LOOKAHEAD": 30})])
def test_tight_rings_are_taken(gpu, monkeypatch, mode, env):
    sc = scene(mode)
    ref = Simulator.from_scene(sc)
    for k, v in env.items():
        monkeypatch.setenv("CC_" + k, str(v))
    sim = Simulator.from_scene(sc)
    for n in (1, 1, 2 * sim.block_steps, 3, sim.block_steps + 1, 40, 1):
        for s in (ref, sim):
            s.simulate(n)
        for x, y in zip(sim.get_state(), ref.get_state()):
            np.testing.assert_array_equal(x, y)
    ref.close()
    sim.close()


@pytest.mark.parametrize("mode,env", [
    (RB, {"GRAPH_STEPS": 10}), (RB, {"LOOKAHEAD": 34}), (RB, {"GRAPH_STEPS": 12, "BUILD_FRAMES": 4}),
    (RF, {"GRAPH_STEPS": 14, "BODY_LANES": 3})])
def test_rings_that_are_too_small_are_refused(gpu, monkeypatch, mode, env):
    for k, v in env.items():
        monkeypatch.setenv("CC_" + k, str(v))
    with pytest.raises(L.ClothCoreError) as e:
        Simulator.from_scene(scene(mode))
    assert e.value.code == L.CC_ERR_INVALID, str(e.value)
