"""A held contact view takes the slots that a launch changed: after every call its first
min(count, M) slots are the oracle's bit for bit, and at the end the whole view, slots past the
count included, is what a world that held none copies from the device."""
import numpy as np
import pytest

from tests.parity import make_pair

pytestmark = pytest.mark.gpu


def check(view, o):
    M = view.shape[1]
    live = np.arange(M)[None, :] < np.minimum(o.contact_counts, M)[:, None]
    for f in ("position_pen", "normal_friction", "indices", "impulses"):
        a, b = np.ascontiguousarray(view[f][live]), np.ascontiguousarray(o.contacts[f][live])
        np.testing.assert_array_equal(a.view(np.uint32), b.view(np.uint32), err_msg=f)


def three(*args, **kw):
    g, o, acts = make_pair(*args, **kw)
    late, _, _ = make_pair(*args, **kw)
    return g, late, o, acts


@pytest.mark.parametrize("shape", [dict(), dict(envs_per_wave=8, split=True, waves=1), dict(envs_per_wave=2, split=False),
                                   dict(placement=1), dict(placement=2)], ids=str)
@pytest.mark.parametrize("substeps", [1, 3])
def test_robots(shape, substeps):
    E = 19
    g, late, o, acts = three("ant", E, 24, seed=5, substeps=substeps, **shape)
    for w in (g, late, o):
        w.step(acts[0])
    view = g.get_contacts(zero_copy=True)
    rng = np.random.default_rng(3)
    for k in range(1, 24):
        if k % 7 == 3:
            mask = (rng.random(E) < 0.4).astype(np.uint8)
            for w in (g, late, o):
                w.reset(mask)
        if k % 5 == 2:
            mask = (rng.random(E) < 0.6).astype(np.uint8)
            mask[:2] = (1, 0)
            for w in (g, late, o):
                w.step_subset(acts[k], mask)
        else:
            for w in (g, late, o):
                w.step(acts[k])
        check(view, o)
    assert view.tobytes() == late.get_contacts(zero_copy=False).tobytes()


@pytest.mark.parametrize("M,extended", [(64, False), (130, True), (200, True), (512, True)])
@pytest.mark.parametrize("pool", [None, "7"])
def test_piles_on_the_ground(monkeypatch, M, extended, pool):
    """Full lists whose slots come into contact and leave it, and raised and lowered counts."""
    if pool:
        monkeypatch.setenv("ZENO_AMD_POOL", pool)
    E = 4
    g, late, o, _ = three("pile", E, 1, seed=6, max_contacts=M, extended_contacts=extended, substeps=2)
    pos = o.positions.copy()
    pos[:, 1:, 2] *= 0.25
    none, zero = np.zeros((E, 0), np.float32), np.zeros_like(o.positions)
    view = g.get_contacts(zero_copy=True)
    for w in (g, late, o):
        w.reset_to_state(pos, o.quaternions.copy(), zero, zero)
    held = 0
    for k in range(24):
        if k in (12, 17):
            counts = np.array([0, M // 2, M, M + 5], np.uint32) if k == 12 else np.full(E, M, np.uint32)
            for w in (g, late):
                w.set_contact_counts(counts)
            o.contact_counts[:] = counts
        before = view.copy()
        for w in (g, late, o):
            w.step(none, substeps=1 + k % 2)
        check(view, o)
        held += int((view.view(np.uint8).reshape(E * M, -1) == before.view(np.uint8).reshape(E * M, -1)).all(1).sum())
    assert held > 0
    assert view.tobytes() == late.get_contacts(zero_copy=False).tobytes()


def test_after_a_capture_and_a_replay():
    E = 7
    g, late, o, _ = three("pile", E, 1, seed=9)
    none = np.zeros((E, 0), np.float32)
    view = g.get_contacts(zero_copy=True)
    for w in (g, late, o):
        w.step(none)
    for w in (g, late):
        w.capture_steps(0, 0, 3)
    for _ in range(3):
        for w in (g, late, o):
            w.step(none)
        check(view, o)
        for w in (g, late):
            w.graph_launch()
        for _ in range(3):
            o.step(none)
        check(view, o)
    assert view.tobytes() == late.get_contacts(zero_copy=False).tobytes()
