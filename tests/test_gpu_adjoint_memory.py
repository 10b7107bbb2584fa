"""CC_ADJ_KEEP_MB bounds the states that a gradient keeps instead of its
checkpoints: at 0 the caller's checkpoint interval alone sets the memory, and
the gradient is the same."""
import numpy as np
import pytest

from simulator_amd import scene as S
from simulator_amd.adjoint import Adjoint
from simulator_amd.simulator import Simulator

from test_gpu_errors import _free_device_bytes

pytestmark = pytest.mark.gpu


def test_kept_states_are_bounded(gpu, monkeypatch):
    sc = S.small(side=128, y0=0.803)
    sim = Simulator.from_scene(sc)
    g = np.random.default_rng(1).normal(size=(sc.n, 3)).astype(np.float32)
    took, out = {}, {}
    for mb in (None, "0", "200", "100"):                 # every state: 118 MB
        if mb is not None:
            monkeypatch.setenv("CC_ADJ_KEEP_MB", mb)
        free = _free_device_bytes()
        adj = Adjoint(sim, 200, 20)
        took[mb] = (free - _free_device_bytes()) / 2**20
        x = adj.forward(sc.pos, None, [900.0, 450.0, 90.0, -0.03, 1.01])
        out[mb] = (x, *adj.backward(g))
        adj.close()
    assert took[None] > 100 and took["200"] > 100, took
    assert took["0"] < 50 and took["100"] < 50, took
    for mb in ("0", "200", "100"):
        for a, b in zip(out[mb], out[None]):
            np.testing.assert_array_equal(a, b)
    sim.close()
