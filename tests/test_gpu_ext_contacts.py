"""Extended-contact mode of the step on the GPU against the CPU oracle, through the C ABI
(zeno_amd_world_set_extended_contacts). The pile's box and capsule pairs go through
narrow_phase.detectCollision in both; discrete outputs are bit-exact and fp32 state within
the contact-rich tolerance of the other multi-step tests.
"""
import numpy as np
import pytest

from tests.parity import compare, gpu_arrays, make_pair, oracle_arrays

pytestmark = pytest.mark.gpu


# One environment per workgroup with M >= 64 runs the narrow phase grouped by geom-type pair
# (every placement, with and without the hash, is covered below); Ant at four environments
# per wave runs it ungrouped.
@pytest.mark.parametrize("name,envs,steps,M,placement,epw", [("pile", 8, 12, 512, None, None),
                                                             ("pile", 4, 8, 512, 2, None),
                                                             ("pile", 4, 8, 512, 0, 1),
                                                             ("pile_hash", 4, 6, 512, None, None),
                                                             ("pile_hash", 2, 4, 512, 2, None),
                                                             ("ant", 16, 20, 128, None, 1),
                                                             ("ant", 16, 20, 64, None, None)])
def test_extended_contacts_parity(name, envs, steps, M, placement, epw):
    g, o, acts = make_pair(name, envs, steps, seed=5, max_contacts=M, placement=placement,
                           envs_per_wave=epw, extended_contacts=True)
    active = 0
    for k in range(steps):
        g.step(acts[k])
        o.step(acts[k])
        compare(gpu_arrays(g), oracle_arrays(o), rtol=1e-4, atol=1e-4)
        live = np.arange(M)[None, :] < np.minimum(o.contact_counts, M)[:, None]
        active += int(((o.contacts["position_pen"][..., 3] >= 0) & live).sum())
    if name != "ant":
        assert active > 0


def test_mode_is_off_by_default_and_switchable():
    g, o, acts = make_pair("pile", 2, 2, seed=6, max_contacts=512)
    g.step(acts[0])
    o.step(acts[0])
    compare(gpu_arrays(g), oracle_arrays(o), rtol=1e-5, atol=1e-6)
    g.set_extended_contacts(True)
    o.extended_contacts = True
    g.step(acts[1])
    o.step(acts[1])
    compare(gpu_arrays(g), oracle_arrays(o), rtol=1e-4, atol=1e-4)


def test_extended_mode_switches_to_the_grouped_shape_and_back():
    """A placement-0 world with a long contact list runs the extended mode in the
    one-environment-per-wave shape without split groups (the type-grouped narrow phase) and
    returns to its creation-time shape when the mode is turned off; both stay on the oracle."""
    g, o, acts = make_pair("pile", 24, 6, seed=8, max_contacts=512)
    if g.modes()["placement"] != 0:
        pytest.skip("the world placed this scene outside LDS")
    base = (g.launch_config()[0], g.waves_per_group(), g.split_groups())
    g.set_extended_contacts(True)
    o.extended_contacts = True
    assert g.launch_config()[0] == 1 and not g.split_groups()
    for k in range(3):
        g.step(acts[k])
        o.step(acts[k])
        compare(gpu_arrays(g), oracle_arrays(o), rtol=1e-4, atol=1e-4)
    g.set_extended_contacts(False)
    o.extended_contacts = False
    assert (g.launch_config()[0], g.waves_per_group(), g.split_groups()) == base
    for k in range(3, 6):
        g.step(acts[k])
        o.step(acts[k])
        compare(gpu_arrays(g), oracle_arrays(o), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("envs,M", [(40, 200), (1300, 200), (1300, 128)])
def test_extended_mode_shape_follows_the_env_count(envs, M):
    """The extended mode's shape, with the model records in LDS for few environments and in HBM
    where that lets more be resident: each stays on the oracle, and turning the mode off restores
    the creation-time shape."""
    g, o, acts = make_pair("pile", envs, 4, seed=9, max_contacts=M)
    base = (g.modes()["placement"], g.launch_config(), g.waves_per_group(), g.split_groups())
    g.set_extended_contacts(True)
    o.extended_contacts = True
    assert g.launch_config()[0] == 1 and not g.split_groups()
    for k in range(4):
        if k == 3:
            g.set_extended_contacts(False)
            o.extended_contacts = False
            assert (g.modes()["placement"], g.launch_config(), g.waves_per_group(), g.split_groups()) == base
        g.step(acts[k])
        o.step(acts[k])
        compare(gpu_arrays(g), oracle_arrays(o), rtol=1e-4, atol=1e-4)


def negative_radii_mjcf(bodies: int = 6) -> str:
    geoms = ('<geom type="sphere" size="-0.3" mass="1"/>', '<geom type="box" size="0.2 0.15 0.1" mass="1"/>',
             '<geom type="capsule" size="-0.25 0.1" mass="1"/>')
    rows = [f'<body name="b{i}" pos="{0.1 * i:.3f} {0.05 * (i % 2):.3f} {0.4 + 0.05 * i:.3f}"><joint type="free"/>{geoms[i % 3]}</body>'
            for i in range(bodies)]
    return '<mujoco><worldbody><geom type="plane" size="20 20 0.1"/>' + "".join(rows) + "</worldbody></mujoco>"


@pytest.mark.parametrize("M", [48, 64, 200])
def test_hits_of_negative_penetration(M):
    """A sphere or capsule of negative radius takes part in hits whose penetration is negative:
    their slots get the point, normal and friction, and neither the matching nor the solve visits
    them."""
    from oracle.oracle import OracleWorld
    from zeno_amd.model import load_model
    from zeno_amd.world import ZenoWorld

    xml = negative_radii_mjcf()
    g = ZenoWorld(mjcf_string=xml, num_envs=3, max_contacts_per_env=M)
    o = OracleWorld(load_model(mjcf_string=xml), 3, max_contacts_per_env=M)
    g.set_extended_contacts(True)
    o.extended_contacts = True
    rng = np.random.default_rng(2)
    state = [x.copy() for x in (o.positions, o.quaternions, o.velocities, o.angular_velocities)]
    state[2][:, 1:, :3] = rng.uniform(-2, 2, (3, 6, 3))
    state[3][:, 1:, :3] = rng.uniform(-3, 3, (3, 6, 3))
    for w in (g, o):
        w.reset_to_state(*state)
    none, seen = np.zeros((3, 0), np.float32), 0
    for k in range(8):
        g.step(none)
        o.step(none)
        pen = o.contacts["position_pen"][..., 3]
        seen += int(((pen < 0) & (pen != -1)).sum())
        compare(gpu_arrays(g), oracle_arrays(o), 0.0, 0.0)
    assert seen > 0


def test_extended_mode_takes_its_own_pool_with_records_in_hbm():
    """Boxes meet the ground in the extended mode alone, so its pool is larger; a world whose model
    records are in HBM switches to it and back."""
    from zeno_amd.scenes import pile_mjcf
    from zeno_amd.world import ZenoWorld

    w = ZenoWorld(mjcf_string=pile_mjcf(64, seed=3), num_envs=6000, max_contacts_per_env=128)
    base = (w.modes()["placement"], w.launch_config())
    assert base[0] == 1
    w.set_extended_contacts(True)
    assert w.modes()["placement"] == 1 and w.launch_config()[1] > base[1][1]
    for _ in range(3):
        w.step(np.zeros((6000, 0), np.float32))
    assert np.isfinite(w.get_body_positions()).all()
    w.set_extended_contacts(False)
    assert (w.modes()["placement"], w.launch_config()) == base
    w.close()
