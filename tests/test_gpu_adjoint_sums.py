"""The gradient's parameter sums over the steps (chunks of 256 in one workgroup
per 256 vertices) and its spring terms added across lanes, bit for bit against
the other ways to compute them: kept states (one sum over all steps) or
checkpoints of 20, four lanes per vertex or one (beyond 98,304 vertices)."""
import numpy as np
import pytest

from test_gpu_adjoint_paths import gradient, scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [255, 256, 257, 513])
@pytest.mark.parametrize("side", [3, 17])
def test_sums_over_many_steps(gpu, side, steps):
    pos, sim, n = scene(side)
    want = gradient(pos, sim, n, steps, steps)
    for a, b in zip(want, gradient(pos, sim, n, steps, 20, True)):
        np.testing.assert_array_equal(a, b)
    sim.close()


@pytest.mark.parametrize("wide,ell", [(False, "1"), (False, "0"), (True, "1")])
def test_four_lanes_equal_one(gpu, monkeypatch, wide, ell):
    monkeypatch.setenv("CC_SPRINGS_ELL", ell)
    out = []
    for total in (0, 98304, 98305):
        pos, sim, n = scene(23, extra=max(total - 23 * 23, 0), wide=wide)
        out.append(gradient(pos, sim, n, 9, 5))
        sim.close()
    for other in out[1:]:
        for a, b in zip(out[0], other):
            np.testing.assert_array_equal(a, b)
