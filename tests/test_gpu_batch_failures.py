"""A launch that fails inside a batch's step, whose cloths run on a stream of
their own beside the bodies: while a block of steps is captured and in single
steps, at every point of a step.  The call reports its own error, the failed
batch can be destroyed, and what runs next on the thread sees nothing of it."""
import numpy as np
import pytest

from simulator_amd import _lib as L
from simulator_amd import batch as B
from simulator_amd import scene as S
from simulator_amd.simulator import Simulator

from test_gpu_batch_refit import instance

pytestmark = pytest.mark.gpu


def scenes():
    return [instance(k, m, mode) for k, (m, mode) in enumerate(
        [(700, L.CC_BODY_REFIT), (300, L.CC_BODY_REBUILD), (50, L.CC_BODY_STATIC)])]


@pytest.mark.parametrize("steps", [16, 1])
def test_failed_launch_in_a_step(gpu, steps):
    scs = scenes()
    sim = Simulator.from_scene(S.small(side=16))
    ref = B.Batch(scs)
    ref.simulate(steps)
    want = [ref.get_state(i) for i in range(len(scs))]
    ref.close()
    failures = 0
    for k in range(64):
        print("steps", steps, "failure", k, flush=True)
        b = B.Batch(scs)
        L.fault_inject(L.CC_FAULT_LAUNCH, k)
        try:
            b.simulate(steps)
            failed = False
        except L.ClothCoreError as e:
            failed = True
            assert e.code == L.CC_ERR_HIP and "injected" in str(e), str(e)
        finally:
            L.fault_inject(L.CC_FAULT_LAUNCH, -1)
        sim.simulate(1)                      # another handle's launch checks
        sim.check_finite()
        b.close()
        failures += failed
        if not failed:
            break
    assert failures == (k if steps == 1 else 64) and failures > 5
    again = B.Batch(scs)
    again.simulate(steps)
    for i, w in enumerate(want):
        for x, y in zip(again.get_state(i), w):
            np.testing.assert_array_equal(x, y)
    again.close()
    sim.close()
