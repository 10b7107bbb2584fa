"""The ways a gradient is computed, against each other bit for bit: the
forward's states kept whole or recomputed from checkpoints (the kept
trajectory's allocation is made to fail), four lanes per vertex or one (the
same cloth alone, and followed by enough loose pinned vertices to pass the
four-lane limit), and springs in fixed-width or merged rows."""
import numpy as np
import pytest

from simulator_amd import _lib as L
from simulator_amd import scene as S
from simulator_amd.adjoint import Adjoint
from simulator_amd.simulator import Simulator

pytestmark = pytest.mark.gpu

CC_FAULT_ALLOC = 1


def scene(side, extra=0, wide=False):
    """A cloth in contact with the sphere, `extra` loose pinned vertices after
    it; wide: mesh springs beside the grid's (rows of more than 12)."""
    sc = S.small(side=side, y0=0.803)
    if wide:
        v4 = np.concatenate([sc.pos, np.ones((sc.n, 1), np.float32)], 1)
        st, be = S.springs_from_mesh(v4, S.grid_faces(side, side))
        sc.springs = [sc.springs[0], sc.springs[1], be]
    pos = np.concatenate([sc.pos, np.zeros((extra, 3), np.float32)]).astype(np.float32)
    springs = [(np.concatenate([r, np.full(extra, r[-1], np.uint32)]).astype(np.uint32), c) for r, c in sc.springs]
    pins = np.concatenate([sc.pins, np.arange(sc.n, sc.n + extra)]).astype(np.uint32)
    return pos, Simulator(pos, springs, sc.body, sc.params, pins), sc.n


def gradient(pos, sim, n, steps, ckpt, fail=False):
    rng = np.random.default_rng(3)
    v0 = np.zeros_like(pos)
    v0[:n] = rng.normal(scale=0.05, size=(n, 3))
    g = np.zeros_like(pos)
    g[:n] = rng.normal(size=(n, 3))
    if fail:
        L.check(L.lib().cc_fault_inject(CC_FAULT_ALLOC, 0))
    try:
        adj = Adjoint(sim, steps, ckpt)
    finally:
        L.lib().cc_fault_inject(CC_FAULT_ALLOC, -1)
    out = []
    for _ in range(2):                                   # a second rollout on the same handle
        x = adj.forward(pos, v0, [900.0, 450.0, 90.0, -0.03, 1.01])
        dth, dv0, dx0 = adj.backward(g)
        out.append((x[:n], dth, dv0[:n], dx0[:n]))
    adj.close()
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    assert all(np.isfinite(a).all() for a in out[0]) and np.any(out[0][1] != 0)
    return out[0]


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("side", [4, 8, 17, 40])
def test_kept_states_equal_checkpoints(gpu, side, wide):
    pos, sim, n = scene(side, wide=wide)
    want = gradient(pos, sim, n, 23, 23)
    for ckpt in (1, 7, 40):
        for fail in (False, True):
            for a, b in zip(want, gradient(pos, sim, n, 23, ckpt, fail)):
                np.testing.assert_array_equal(a, b)
    sim.close()


@pytest.mark.parametrize("ell", ["1", "0"])
def test_one_lane_equals_four(gpu, monkeypatch, ell):
    monkeypatch.setenv("CC_SPRINGS_ELL", ell)
    pos, sim, n = scene(40)
    want = gradient(pos, sim, n, 12, 5)
    sim.close()
    pos, sim, n = scene(40, extra=65537 - n)
    for a, b in zip(want, gradient(pos, sim, n, 12, 5)):
        np.testing.assert_array_equal(a, b)
    sim.close()
