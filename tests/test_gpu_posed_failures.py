"""Replacing a body's vertices where an allocation or a launch fails, at every
point of the call.  Afterwards the simulator either steps over a whole tree or
refuses to (CC_ERR_INVALID): blocks of steps recorded before must not be
replayed over buffers that the call has freed, nor tables of one tree used with
those of another.  A static body whose four-wide records do not fit is walked
in the binary form, with the same results.  The next replacement that succeeds
makes all of it good: bit for bit a simulator that saw no failure."""
import numpy as np
import pytest

from simulator_amd import _lib as L
from simulator_amd import scene as S
from simulator_amd.simulator import Simulator

from test_gpu_posed import scene, turned

pytestmark = pytest.mark.gpu


def stepped(body):
    sim = Simulator.from_scene(scene(body))
    sim.simulate(2 * sim.block_steps + 1)                # blocks over the body as created
    return sim


def fails_at(sim, v, kind, k):
    L.fault_inject(kind, k)
    try:
        sim.set_body_vertices(v)
    except L.ClothCoreError as e:
        assert e.code == (L.CC_ERR_ALLOC if kind == L.CC_FAULT_ALLOC else L.CC_ERR_HIP), str(e)
        return True
    finally:
        L.fault_inject(kind, -1)
    return False


def follow(a, b, steps):
    for n in steps:
        for s in (a, b):
            s.simulate(n)
        for x, y in zip(a.get_state(), b.get_state()):
            np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("up", ["1", "0"])
@pytest.mark.parametrize("kind", [L.CC_FAULT_ALLOC, L.CC_FAULT_LAUNCH])
@pytest.mark.parametrize("mode", [L.CC_BODY_STATIC, L.CC_BODY_REFIT, L.CC_BODY_REBUILD])
def test_a_failed_replacement_is_recovered_from(gpu, mode, kind, up, monkeypatch):
    monkeypatch.setenv("CC_REBUILD_BOTTOM_UP", up)
    body = S.capsules(16, 4, 3, mode)
    v = np.ascontiguousarray(body.verts * np.float32([1.0, 1.0, 0.8]))   # another topology
    for k in range(200):
        print("mode", mode, "kind", kind, "levels", up, "failure", k, flush=True)
        sim, ref = stepped(body), stepped(body)
        failed = fails_at(sim, v, kind, k)
        if failed:
            try:
                sim.simulate(sim.block_steps + 1)
                ref.simulate(ref.block_steps + 1)
            except L.ClothCoreError as e:
                assert e.code == L.CC_ERR_INVALID and mode != L.CC_BODY_REBUILD, str(e)
            sim.set_body_vertices(v)
        ref.set_body_vertices(v)
        sim.set_frame(ref.frame)
        sim.set_state(*ref.get_state())
        assert sim.bvh_width() == ref.bvh_width()
        a, b = sim.bvh_export(), ref.bvh_export()
        for key in a:
            np.testing.assert_array_equal(a[key], b[key], err_msg=key)
        follow(sim, ref, (1, sim.block_steps, 2))
        sim.close()
        ref.close()
        if not failed:
            break
    assert not failed and k > 0


def test_a_static_body_without_wide_records_is_walked_in_the_binary_form(gpu):
    body = S.capsules(16, 4, 3, L.CC_BODY_STATIC)
    v = turned(body.verts, 0.05)
    sim, ref = stepped(body), stepped(body)
    assert fails_at(sim, v, L.CC_FAULT_ALLOC, 1)         # 0: the pinned memory
    ref.set_body_vertices(v)
    assert sim.bvh_width()[0] == 2 and ref.bvh_width()[0] == 4
    follow(sim, ref, (sim.block_steps, 3))
    sim.close()
    ref.close()


def test_the_binary_walk_stays_where_the_records_cannot_be_folded(gpu):
    body = S.capsules(16, 4, 3, L.CC_BODY_STATIC)
    v = turned(body.verts, 0.05)
    sim, ref = stepped(body), stepped(body)
    for s in (sim, ref):
        s.set_bvh_width(2)
        s.set_body_vertices(v)
    L.fault_inject(L.CC_FAULT_LAUNCH, 0)
    try:
        with pytest.raises(L.ClothCoreError):
            sim.set_bvh_width(4)
    finally:
        L.fault_inject(L.CC_FAULT_LAUNCH, -1)
    assert sim.bvh_width()[0] == 2
    follow(sim, ref, (2,))
    for s in (sim, ref):
        s.set_bvh_width(4)
        assert s.bvh_width()[0] == 4
    follow(sim, ref, (sim.block_steps, 1))
    sim.close()
    ref.close()
