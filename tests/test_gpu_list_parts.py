"""Worlds whose device memory held the scratch contact lists of some environments only: a launch
runs in parts of that many, one after another. ZENO_AMD_LIST_ENVS starts a world there; everything
that a call hands out, per-environment arrays of every kind, against the oracle bit for bit."""
import numpy as np
import pytest

from tests.parity import compare, gpu_arrays, make_pair, oracle_arrays
from tests.test_gpu_graph import DeviceBuffer

pytestmark = pytest.mark.gpu


def check(g, o, views=None):
    arrays = gpu_arrays(g)
    compare(arrays, oracle_arrays(o), 0.0, 0.0)
    for name, view in (views or {}).items():
        np.testing.assert_array_equal(view.view(np.uint32), np.ascontiguousarray(arrays[name]).view(np.uint32), err_msg=name)


@pytest.mark.parametrize("part", [1, 3, 8, 12])
@pytest.mark.parametrize("name,shape", [("ant", dict()), ("ant", dict(envs_per_wave=4, split=True, waves=4, substeps=2)),
                                        ("cartpole", dict(envs_per_wave=8)), ("pile", dict(max_contacts=130, extended_contacts=True))],
                         ids=str)
@pytest.mark.parametrize("held", [False, True])
def test_launches_in_parts(monkeypatch, part, name, shape, held):
    monkeypatch.setenv("ZENO_AMD_LIST_ENVS", str(part))
    E, K = 19, 13
    g, o, acts = make_pair(name, E, K, seed=7, **shape)
    views = dict(positions=g.get_body_positions(zero_copy=True), velocities=g.get_body_velocities(zero_copy=True),
                 accelerations=g.get_body_accelerations(zero_copy=True), quaternions=g.get_body_quaternions(zero_copy=True),
                 angular_velocities=g.get_body_angular_velocities(zero_copy=True), joint_positions=g.get_joint_positions(zero_copy=True),
                 joint_velocities=g.get_joint_velocities(zero_copy=True), joint_torques=g.get_joint_forces(zero_copy=True),
                 observations=g.get_observations(zero_copy=True)) if held else None
    if held:
        g.get_contacts(zero_copy=True)
    rng = np.random.default_rng(4)
    for k in range(K):
        if k in (5, 9):
            mask = (rng.random(E) < 0.4).astype(np.uint8)
            g.reset(mask)
            o.reset(mask)
        if k % 4 == 2:
            mask = (rng.random(E) < 0.6).astype(np.uint8)
            mask[:2] = (1, 0)
            g.step_subset(acts[k], mask)
            o.step_subset(acts[k], mask)
        else:
            g.step(acts[k])
            o.step(acts[k])
        check(g, o, views)


def test_schedules_in_parts(monkeypatch):
    monkeypatch.setenv("ZENO_AMD_LIST_ENVS", "5")
    E, K = 13, 70
    g, o, acts = make_pair("ant", E, K, seed=8)
    buf = DeviceBuffer(np.ascontiguousarray(acts, np.float32).reshape(-1))
    try:
        g.capture_steps(buf.ptr.value, E * g.action_dim * 4, K)
        for _ in range(2):
            g.graph_launch()
            for k in range(K):
                o.step(acts[k])
            check(g, o)
            g.step(acts[0])
            o.step(acts[0])
        counts = o.contact_counts.copy()
        g.set_contact_counts(counts)
        g.graph_launch()
        for k in range(K):
            o.step(acts[k])
        check(g, o)
    finally:
        g.release_graph()
        buf.free()


def test_memory_of_the_scratch_lists(monkeypatch):
    """Two lists of 64 B a slot for as many environments as a part holds, a third from the first
    masked step on."""
    def used(part):
        monkeypatch.setenv("ZENO_AMD_LIST_ENVS", str(part))
        g, _, acts = make_pair("ant", 40, 1, seed=2)
        before = g.gpu_memory_usage
        g.close()
        return before

    assert used(40) - used(10) == 30 * 2 * 64 * 64
