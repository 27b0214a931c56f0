"""Counts the host raises expose slots that no sort has covered, and the next step of every
environment sorts its list once (zeno_amd_world_set_contact_counts). That step may be an eager one
after a capture, the first of a replayed schedule, or, for an environment that a step mask holds
back, a later one: each against the oracle, which sorts every list in every step."""
import numpy as np
import pytest

from tests.parity import compare, gpu_arrays, make_pair, oracle_arrays
from tests.test_gpu_graph import DeviceBuffer

pytestmark = pytest.mark.gpu

E, M = 5, 200
NONE = np.zeros((E, 0), np.float32)


def exposed(**shape):
    """A list filled and sorted, then reset and appended to from slot 0: the slots behind the new
    ones hold the old list's end. Raising the counts to M exposes them, out of order."""
    g, o, _ = make_pair("pile", E, 1, seed=21, max_contacts=M, **shape)
    for w in (g, o):
        for _ in range(5):
            w.step(NONE)
        w.reset()
        w.step(NONE)
    counts = np.full(E, M, np.uint32)
    counts[1] = M + 7
    keys = o.contacts["indices"][..., :2].astype(np.int64)
    keys = np.sort(keys, axis=-1) @ np.array([1 << 16, 1])
    assert (o.contact_counts < M).all() and (np.diff(keys, axis=1) < 0).any(1).all()
    return g, o, counts


def raise_counts(g, o, counts):
    g.set_contact_counts(counts)
    o.contact_counts[:] = counts


def check(g, o):
    compare(gpu_arrays(g), oracle_arrays(o), 0.0, 0.0)


SHAPES = [dict(), dict(placement=1), dict(placement=3)]


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("steps", [1, 70])
def test_a_capture_leaves_the_sort_to_the_next_step(shape, steps):
    g, o, counts = exposed(**shape)
    raise_counts(g, o, counts)
    g.capture_steps(0, 0, steps)
    for _ in range(2):
        g.step(NONE)
        o.step(NONE)
        check(g, o)
    g.graph_launch()
    for _ in range(steps):
        o.step(NONE)
    check(g, o)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("held", [False, True])
@pytest.mark.parametrize("steps,substeps", [(1, 1), (3, 2), (70, 1)])
def test_a_replayed_schedule_sorts_first(shape, held, steps, substeps):
    g, o, counts = exposed(**shape)
    view = g.get_contacts(zero_copy=True) if held else None
    g.capture_steps(0, 0, steps, substeps)
    g.step(NONE)  # another dt than the schedule's
    o.step(NONE)
    for w in (g, o):
        w.reset()
        w.step(NONE)
    raise_counts(g, o, counts)
    for _ in range(3):
        g.graph_launch()
        for _ in range(steps):
            o.step(NONE, substeps=substeps)
        if held:
            live = np.minimum(o.contact_counts, M)
            for e in range(E):
                assert view[e, : live[e]]["indices"].tobytes() == o.contacts[e, : live[e]]["indices"].tobytes()
        check(g, o)


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_a_masked_step_leaves_the_sort_of_those_it_holds_back(shape):
    g, o, counts = exposed(**shape)
    raise_counts(g, o, counts)
    for mask in ([1, 0, 0, 1, 0], [0, 1, 0, 1, 0]):  # environments 2 and 4 are held back twice
        mask = np.array(mask, np.uint8)
        g.step_subset(NONE, mask)
        o.step_subset(NONE, mask)
        check(g, o)
    for _ in range(2):
        g.step(NONE)
        o.step(NONE)
        check(g, o)
    # Every environment advanced by masks alone, then a replay.
    for w in (g, o):
        w.reset()
        w.step(NONE)
    raise_counts(g, o, counts)
    g.capture_steps(0, 0, 2)
    for mask in ([1, 1, 0, 0, 0], [0, 0, 1, 1, 0]):
        mask = np.array(mask, np.uint8)
        g.step_subset(NONE, mask)
        o.step_subset(NONE, mask)
    g.graph_launch()
    for _ in range(2):
        o.step(NONE)
    check(g, o)
