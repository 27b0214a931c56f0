"""The contact pool: the contact list in HBM and its valid slots in LDS (make_env_pool), against
the oracle bit for bit. ZENO_AMD_POOL shrinks the pool so that some or all environments have more
valid slots than it holds and run their contact solve out of HBM; lists grow, fill, are reset, held
back by a step mask and sorted meanwhile."""
import numpy as np
import pytest

from tests.parity import compare, gpu_arrays, make_pair, oracle_arrays

pytestmark = pytest.mark.gpu


def check(g, o, what):
    compare(gpu_arrays(g), oracle_arrays(o), 0.0, 0.0)


@pytest.mark.parametrize("pool", [1, 7, 33, 64])
@pytest.mark.parametrize("shape", [
    dict(placement=1), dict(envs_per_wave=1, split=False), dict(envs_per_wave=1, split=True, waves=1),
    dict(envs_per_wave=2, split=True, waves=1), dict(placement=1, substeps=3), dict(placement=1, extended_contacts=True),
    dict(envs_per_wave=2, split=True, waves=1, substeps=2),
], ids=lambda s: "-".join(f"{k}{int(v)}" for k, v in s.items()))
def test_pile_pools(monkeypatch, pool, shape):
    """64 bodies: lists of 64 slots, full of ground pairs after one step; environments with a fifth
    to all of their spheres and capsules (some forty slots) on the ground."""
    monkeypatch.setenv("ZENO_AMD_POOL", str(pool))
    g, o, acts = make_pair("pile", 5, 1, seed=3, **shape)
    pos = o.positions.copy()
    geoms = o.model["geoms"][1:]
    height = geoms["pos_size0"][:, 3] + np.where(geoms["type_body"][:, 0] == 1, geoms["params"][:, 0], 0.0)
    for e in range(5):
        pos[e, 1:, 2] = height - 0.002 + np.where(np.arange(64) % 5 < e, 0.0, 1.0)
    for w in (g, o):
        w.reset_to_state(pos, o.quaternions.copy(), np.zeros_like(pos), np.zeros_like(pos))
    most = 0
    for k in range(9):
        g.step(np.zeros((5, 0), np.float32))
        o.step(np.zeros((5, 0), np.float32))
        most = max(most, (o.contacts["position_pen"][..., 3] >= 0).sum(1).max())
        check(g, o, k)
    assert most > min(pool, 25), most


@pytest.mark.parametrize("pool,epw", [(2, 4), (2, 8), (24, 8), (64, 4)])
def test_robot_pools_through_resets_and_masks(monkeypatch, pool, epw):
    """Ant: lists that start anew at every reset, and environments held back by a mask whose solver
    history advances while their visible list stays."""
    monkeypatch.setenv("ZENO_AMD_POOL", str(pool))
    E = 2 * epw + 3
    g, o, acts = make_pair("ant", E, 24, seed=5, envs_per_wave=epw, split=True, waves=1)
    rng = np.random.default_rng(9)
    for k in range(24):
        if k in (7, 15):
            mask = (rng.random(E) < 0.4).astype(np.uint8)
            g.reset(mask)
            o.reset(mask)
        if k % 5 == 3:
            mask = (rng.random(E) < 0.6).astype(np.uint8)
            mask[0] = 1
            mask[1] = 0
            g.step_subset(acts[k], mask)
            o.step_subset(acts[k], mask)
        else:
            g.step(acts[k])
            o.step(acts[k])
        if k % 6 == 5:
            check(g, o, k)


@pytest.mark.parametrize("m", [1, 5, 63, 65, 130, 200])
def test_list_lengths(monkeypatch, m):
    """List lengths around the 64-slot words of the pool's masks, the pool one slot short."""
    monkeypatch.setenv("ZENO_AMD_POOL", str(max(m - 1, 1)))
    for shape in (dict(placement=1), dict(envs_per_wave=1, split=True, waves=1)):
        g, o, acts = make_pair("pile", 3, 1, seed=8, max_contacts=m, **shape)
        pos = o.positions.copy()
        pos[:, 1:, 2] *= 0.3
        for w in (g, o):
            w.reset_to_state(pos, o.quaternions.copy(), np.zeros_like(pos), np.zeros_like(pos))
        for k in range(9):
            g.step(np.zeros((3, 0), np.float32))
            o.step(np.zeros((3, 0), np.float32))
        check(g, o, m)
        # Lowered counts: slots come back whose order no sort has covered, and appends land below M.
        low = np.array([0, m // 2, m], np.uint32)
        g.set_contact_counts(low)
        o.contact_counts[:] = low
        for k in range(3):
            g.step(np.zeros((3, 0), np.float32))
            o.step(np.zeros((3, 0), np.float32))
        check(g, o, m)
