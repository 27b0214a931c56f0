"""The workloads this library's speed is measured on: what its users have it do, through its
public entry points.

Six kinds, each over the range of sizes it is used at:

  env       the reinforcement-learning loop: one call steps every environment and returns the
            observations. Small vector environments take their actions as numpy arrays through
            ZenoEnv; large ones take them from a policy on the same GPU (torch tensors,
            ZenoWorld.step_device). `substeps` is the frame skip; `reset_every` resets every
            n-th environment before the step, another n-th each time, as auto-reset does when
            episodes end.
  rollout   a fixed schedule of device-resident actions replayed as a graph (model-predictive
            sampling, replay evaluation), then the whole state read back.
  pile      free rigid bodies on a plane: a frame of several substeps, then the poses a viewer
            or a camera model reads.
  pile_ext  the same with box and capsule contacts switched on and long contact lists.
  hash      scenes of more than 512 geoms, whose broad phase is the spatial hash: a pile of free
            bodies, or balls on a static terrain.
  collide   the batched narrow phase on its own, on device or host arrays.

Every state is a running simulation: worlds are stepped past their start in prepare(), because
contact lists fill within the first steps and a user's loop spends its time after that.
"""
import functools
import math

import numpy as np
import torch

from zeno_amd import _lib
from zeno_amd.collision import COLLIDER_DTYPE, detect_collisions
from zeno_amd.env import ZenoEnv
from zeno_amd.model import load_model
from zeno_amd.scenes import ASSETS, pile_initial_state, pile_mjcf, terrain_mjcf
from zeno_amd.world import ZenoWorld

ROBOTS = ("pendulum", "cartpole", "reacher", "pusher", "hopper", "walker", "cheetah", "swimmer", "ant", "humanoid")
ACTION_SETS = 16     # different action arrays that a state cycles through
SETTLE_ENV = 8       # steps before the first pass of a robot world
PILE_XY = (-1.0, 1.0)


def listed():
    return [
        # A single Gym environment driven from Python: pure call latency.
        {"name": "pendulum_env_1", "kind": "env", "robot": "pendulum", "envs": 1, "substeps": 1, "actions": "host", "reset_every": 0},
        # The benchmark's 1024 environments on the smallest articulated scene with a slider.
        {"name": "cartpole_env_1024", "kind": "env", "robot": "cartpole", "envs": 1024, "substeps": 1, "actions": "host", "reset_every": 0},
        # A vector environment of an odd size whose episodes end at different times.
        {"name": "walker_env_3001_resets", "kind": "env", "robot": "walker", "envs": 3001, "substeps": 1, "actions": "host", "reset_every": 64},
        # The headline configuration, as an RL loop sees it.
        {"name": "ant_env_4096", "kind": "env", "robot": "ant", "envs": 4096, "substeps": 1, "actions": "host", "reset_every": 0},
        # The headline configuration as a replayed action schedule.
        {"name": "ant_rollout_4096x32", "kind": "rollout", "robot": "ant", "envs": 4096, "steps": 32, "substeps": 1},
        # A large batch fed by a policy on the GPU: more environments than are resident at once.
        {"name": "ant_env_32768", "kind": "env", "robot": "ant", "envs": 32768, "substeps": 1, "actions": "device", "reset_every": 0},
        # The largest shipped robot at its benchmark size.
        {"name": "humanoid_env_16384", "kind": "env", "robot": "humanoid", "envs": 16384, "substeps": 1, "actions": "device", "reset_every": 0},
        # The usual frame skip of the humanoid tasks, an odd count.
        {"name": "humanoid_skip5_2501", "kind": "env", "robot": "humanoid", "envs": 2501, "substeps": 5, "actions": "host", "reset_every": 0},
        # The benchmark's rigid pile: frames of eight substeps.
        {"name": "pile_8192", "kind": "pile", "bodies": 64, "envs": 8192, "substeps": 8},
        # Box and capsule contacts with the long lists they need.
        {"name": "pile_ext_8192", "kind": "pile_ext", "bodies": 64, "envs": 8192, "substeps": 2, "max_contacts": 512},
        # A crowd of 600 free bodies under the spatial hash.
        {"name": "hash_pile_2048", "kind": "hash", "scene": "pile", "bodies": 600, "envs": 2048, "substeps": 4},
        # The batched narrow phase on a large mixed batch.
        {"name": "collide_8m", "kind": "collide", "pairs": 1 << 23, "where": "device"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["env"] * 5 + ["rollout", "rollout", "pile", "pile", "pile_ext", "hash", "collide", "collide"])
    if kind == "env":
        actions = rng.choice(["host", "device"])
        return {"kind": kind, "robot": rng.choice(ROBOTS), "envs": _log_int(rng, 1, 12000 if actions == "host" else 24000),
                "substeps": rng.choice([1, 1, 1, 2, 4, 5]), "actions": actions, "reset_every": rng.choice([0, 0, 16, 100])}
    if kind == "rollout":
        return {"kind": kind, "robot": rng.choice(ROBOTS), "envs": _log_int(rng, 16, 4096), "steps": rng.randint(2, 24),
                "substeps": rng.choice([1, 1, 2])}
    if kind == "pile":
        return {"kind": kind, "bodies": rng.randint(6, 64), "envs": _log_int(rng, 16, 8192), "substeps": rng.randint(1, 8)}
    if kind == "pile_ext":
        return {"kind": kind, "bodies": rng.randint(12, 64), "envs": _log_int(rng, 16, 4096), "substeps": rng.randint(1, 2),
                "max_contacts": rng.choice([64, 128, 200, 256, 384, 512])}
    if kind == "hash":
        scene = rng.choice(["pile", "terrain"])
        return {"kind": kind, "scene": scene, "bodies": rng.randint(530, 900) if scene == "pile" else rng.randint(4, 24),
                "envs": _log_int(rng, 16, 1024), "substeps": rng.randint(1, 3)}
    where = rng.choice(["device", "host"])
    return {"kind": kind, "pairs": _log_int(rng, 100, 6000000 if where == "device" else 60000), "where": where}


# ---- sizes ---------------------------------------------------------------------------------
def _scene(case):
    """(mjcf path, mjcf string) of a case's scene; the piles' shapes follow from their body count."""
    if case["kind"] in ("env", "rollout"):
        return str(ASSETS / (case["robot"] + ".xml")), None
    if case["kind"] == "hash" and case["scene"] == "terrain":
        return None, terrain_mjcf(case["bodies"], seed=case["bodies"])
    return None, pile_mjcf(case["bodies"], seed=case["bodies"], xy=_xy(case))


def _xy(case):
    if case["kind"] != "hash":
        return PILE_XY
    # The 600 bodies of the benchmark's hash pile lie over 16 x 16; others at that density.
    return (-1.0, 6.0) if case["scene"] == "terrain" else (-3.0, -3.0 + 16.0 * math.sqrt(case["bodies"] / 600.0))


@functools.lru_cache(maxsize=64)
def _model_of(path, xml):
    return load_model(mjcf_path=path, mjcf_string=xml)


def work(case):
    """The state of every environment is read once and written once per call (a rollout's calls
    are its steps taken together), actions are read, and what the caller gets back is written
    once more. Operations: about 250 per joint constraint and 150 per contact slot and solver
    iteration, 150 per body, 12 per candidate pair, each substep."""
    if case["kind"] == "collide":
        return {"bytes": 192 * case["pairs"], "flops": 250 * case["pairs"]}
    m = _model_of(*_scene(case))
    E, B, J, N, M = case["envs"], m["num_bodies"], m["num_joints"], m["num_constraints"], case.get("max_contacts", 64)
    steps = case.get("steps", 1)
    state = 144 * B + 12 * J + 8 * N + 128 * M + 8 + 4 * m["obs_dim"]
    back = 4 * m["obs_dim"] if case["kind"] == "env" else 64 * B + 4 * m["obs_dim"] if case["kind"] == "rollout" else 32 * B
    pairs = m["num_pairs"] if m["num_geoms"] <= 512 else 16 * m["num_geoms"]
    ops = 4 * (250 * N + 150 * min(M, 16)) + 150 * B + 12 * pairs
    return {"bytes": E * (state + back + 4 * m["num_actuators"] * steps), "flops": E * steps * case["substeps"] * ops}


def tolerance(case):
    """Bit for bit: the library's contract is the reference's fp32 operations in the reference's
    order, state and discrete outputs alike, and its tests hold the GPU to that."""
    return "exact"


# ---- states --------------------------------------------------------------------------------
def _action_sets(case, seed, action_dim):
    rng = np.random.default_rng([seed, 1])
    n = case["steps"] if case["kind"] == "rollout" else ACTION_SETS
    return rng.uniform(-1.0, 1.0, (n, case["envs"], action_dim)).astype(np.float32)


def _start_state(case, seed, model):
    """Poses of the first pass: robots start from the scene's pose turned by small random body
    rotations and lifts (reset noise); piles from random drops."""
    if case["kind"] in ("pile", "pile_ext", "hash"):
        return pile_initial_state(model, case["envs"], seed, xy=_xy(case))
    E, B = case["envs"], model["num_bodies"]
    rng = np.random.default_rng([seed, 2])
    pos = np.broadcast_to(model["init_positions"], (E, B, 4)).copy()
    quat = np.broadcast_to(model["init_quaternions"], (E, B, 4)).copy()
    vel = np.zeros((E, B, 4), np.float32)
    ang = np.zeros((E, B, 4), np.float32)
    if case["robot"] not in FIXED_BASE:
        pos[:, 1:, 2] += rng.uniform(0.0, 0.1, (E, 1)).astype(np.float32)
    vel[:, 1:, :3] = rng.uniform(-0.05, 0.05, (E, B - 1, 3))
    ang[:, 1:, :3] = rng.uniform(-0.1, 0.1, (E, B - 1, 3))
    return pos, quat, vel, ang


FIXED_BASE = ("pendulum", "cartpole", "reacher", "pusher")


def prepare(case, seed):
    if case["kind"] == "collide":
        return _prepare_collide(case, seed)
    path, xml = _scene(case)
    model = _model_of(path, xml)
    kw = dict(mjcf_path=path, mjcf_string=xml, num_envs=case["envs"], max_contacts_per_env=case.get("max_contacts", 64))
    s = {"case": case, "pass": 0}
    if case["kind"] == "env" and case["actions"] == "host":
        s["env"] = ZenoEnv(substeps=case["substeps"], **kw)
        w = s["env"].world
    else:
        w = ZenoWorld(substeps=case["substeps"], **kw)
    s["world"] = w
    if case["kind"] == "pile_ext":
        w.set_extended_contacts(True)
    w.reset_to_state(*_start_state(case, seed, model))
    none = np.zeros((case["envs"], w.action_dim), np.float32)
    if case["kind"] in ("env", "rollout"):
        acts = _action_sets(case, seed, w.action_dim)
        for k in range(SETTLE_ENV):
            w.step(acts[k % len(acts)])
        if case["kind"] == "rollout":
            s["acts"] = torch.from_numpy(acts).cuda()
            torch.cuda.synchronize()  # the world steps on a stream of its own
            w.capture_steps(s["acts"].data_ptr(), acts[0].nbytes, len(acts))
        elif case["actions"] == "device":
            s["acts"] = torch.from_numpy(acts).cuda()
            torch.cuda.synchronize()
        else:
            s["acts"] = acts
        if case.get("reset_every"):
            n = case["reset_every"]
            s["masks"] = [(np.arange(case["envs"]) % n == k).astype(np.uint8) for k in range(min(n, ACTION_SETS))]
    else:
        # The bodies reach the ground: 2.25 m take 0.7 s of 2 ms steps.
        for _ in range(350):
            w.step(none, substeps=1)
        s["acts"] = none
    w.synchronize()
    return s


class _View(np.ndarray):
    """A view of a world's host mirror that keeps the world open, as the variable that holds the
    world does in a user's program."""


def _held(world, **views):
    out = {}
    for name, view in views.items():
        out[name] = view.view(_View)
        out[name].world = world
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "collide":
        return _run_collide(state)
    w = state["world"]
    k = state["pass"]
    state["pass"] = k + 1
    if kind == "env":
        if case["reset_every"]:
            w.reset(state["masks"][k % len(state["masks"])])
        a = state["acts"][k % len(state["acts"])]
        if case["actions"] == "host":
            obs, rewards, dones, _ = state["env"].step(a)
            return {"observations": obs, "rewards": rewards, "dones": dones}
        w.step_device(a.data_ptr())
        return _held(w, observations=w.get_observations(zero_copy=True))
    if kind == "rollout":
        w.graph_launch()
        return _held(w, observations=w.get_observations(zero_copy=True), positions=w.get_body_positions(),
                     quaternions=w.get_body_quaternions(), velocities=w.get_body_velocities(),
                     angular_velocities=w.get_body_angular_velocities())
    w.step(state["acts"])
    return _held(w, positions=w.get_body_positions(), quaternions=w.get_body_quaternions())


# ---- the batched narrow phase --------------------------------------------------------------
def _collide_operands(case, seed, device):
    """Uniformly mixed spheres, capsules, boxes and planes, about a third of the pairs in contact."""
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    sides = []
    for _ in range(2):
        n = case["pairs"]
        r = torch.zeros(n, 16, device=device)
        r.view(torch.int32)[:, 0] = torch.randint(0, 4, (n,), generator=g, device=device, dtype=torch.int32)
        r[:, 1:4] = 0.05 + 0.55 * torch.rand(n, 3, generator=g, device=device)
        r[:, 8:11] = -0.7 + 1.4 * torch.rand(n, 3, generator=g, device=device)
        q = torch.randn(n, 4, generator=g, device=device)
        r[:, 12:16] = q / q.norm(dim=1, keepdim=True)
        sides.append(r)
    return sides


def _prepare_collide(case, seed):
    s = {"case": case, "lib": _lib.load()}
    if case["where"] == "device":
        s["a"], s["b"] = _collide_operands(case, seed, "cuda")
        s["out"] = torch.empty(case["pairs"], 16, device="cuda")
    else:
        a, b = _collide_operands(case, seed, "cpu")
        s["a"], s["b"] = (x.numpy().view(COLLIDER_DTYPE).reshape(-1) for x in (a, b))
    return s


def _run_collide(state):
    if state["case"]["where"] == "host":
        r = detect_collisions(state["a"], state["b"])
        return {f: r[f] for f in ("point", "penetration", "normal", "valid", "local_a", "local_b")}
    out = state["out"]
    rc = state["lib"].zeno_amd_detect_collisions(state["a"].data_ptr(), state["b"].data_ptr(), state["case"]["pairs"],
                                                 out.data_ptr(), torch.cuda.current_stream().cuda_stream)
    if rc != 0:
        raise RuntimeError(f"detect_collisions: {rc}: {_lib.last_error()}")
    return {"point": out[:, 0:3], "penetration": out[:, 3], "normal": out[:, 4:7], "valid": out.view(torch.int32)[:, 7],
            "local_a": out[:, 8:12], "local_b": out[:, 12:16]}


# ---- the same in 64 bits -------------------------------------------------------------------
def exact(case, seed):
    """The batched narrow phase, and the robots without ground contact (pendulum, cartpole), in
    64 bits. The other worlds have no such value: whether a slot of the list is in contact, and
    with it the state some steps on, turns on the last bits of the poses."""
    if case["kind"] == "collide":
        return _exact_collide(case, seed)
    if case["kind"] == "env" and case["robot"] in ("pendulum", "cartpole") and not case["reset_every"]:
        out = {"observations": _exact_observations(case, seed)}
        if case["actions"] == "host":
            out.update(rewards=None, dones=None)
        return out
    return None


def _dot(a, b):
    return (a * b).sum(-1, keepdim=True)


def _rotate(v, q):
    u, w = q[..., :3], q[..., 3:4]
    t = torch.linalg.cross(u, v, dim=-1)
    return v + 2.0 * (w * t + torch.linalg.cross(u, t, dim=-1))


def _qmul(a, b):
    v = a[..., 3:] * b[..., :3] + b[..., 3:] * a[..., :3] + torch.linalg.cross(a[..., :3], b[..., :3], dim=-1)
    return torch.cat([v, a[..., 3:] * b[..., 3:] - _dot(a[..., :3], b[..., :3])], -1)


def _conj(q):
    return torch.cat([-q[..., :3], q[..., 3:]], -1)


def _unit(v):
    return v / v.norm(dim=-1, keepdim=True).clamp_min(1e-300)


def _exact_observations(case, seed):
    """Joint-space observations after the settling steps and one pass: position-based dynamics of
    the scene's joints, one constraint after another, without contacts."""
    path, xml = _scene(case)
    m = _model_of(path, xml)
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def t64(x):
        return torch.as_tensor(np.asarray(x, np.float64), device=dev)

    pos, quat, vel, ang = (t64(x) for x in _start_state(case, seed, m))
    pos, vel, ang = pos[..., :3].clone(), vel[..., :3].clone(), ang[..., :3].clone()
    quat = quat.clone()
    im, com = t64(m["inv_mass_inertia"]), t64(m["bodies"]["com_offset"][:, :3])
    inv_m, inv_i = im[:, :1], im[:, 1:]
    moves = (im[:, 0] >= 1e-8)[:, None]
    kinematic = [b for b in range(m["num_bodies"]) if int(m["bodies"]["params"][b, 1]) == 1]
    g = t64(m["gravity"])
    E, J = case["envs"], m["num_joints"]
    acts = _action_sets(case, seed, m["num_actuators"])
    lam = torch.zeros(E, m["num_constraints"], dtype=torch.float64, device=dev)
    tau = torch.zeros(E, J, dtype=torch.float64, device=dev)
    joints, obs = m["joints"], None

    def turn(b, axis, sign):  # orientation of body b moved by a rotation vector in its own inertia
        d = torch.cat([axis * inv_i[b], torch.zeros_like(axis[..., :1])], -1)
        quat[:, b] = _unit(quat[:, b] + sign * 0.5 * _qmul(d, quat[:, b]))

    calls = [acts[k % len(acts)] for k in range(SETTLE_ENV)] + [acts[0]]
    dt = np.float64(np.float32(m["timestep"])) / case["substeps"]
    for a in calls:
        for _ in range(case["substeps"]):
            lam *= 0.8
            for k in range(m["num_actuators"]):
                p, p2 = m["actuators"]["params"][k], m["actuators"]["params2"][k]
                u = t64(a[:, k]).clamp(float(p[1]), float(p[2])) * float(p[3])
                tau[:, int(p[0])] = u.clamp(float(p2[0]), float(p2[1]))
            force = torch.where(moves, g / inv_m.clamp_min(1e-30), torch.zeros_like(g)).expand(E, -1, 3).clone()
            torque = torch.linalg.cross(_rotate(com.expand(E, -1, 3), quat), force, dim=-1)
            for b in kinematic:
                pos[:, b] += vel[:, b] * dt
                w = torch.cat([ang[:, b] * dt * 0.5, torch.zeros_like(ang[:, b, :1])], -1)
                quat[:, b] = _unit(quat[:, b] + _qmul(w, quat[:, b]))
            pos0, quat0 = pos.clone(), quat.clone()
            for j in range(J):
                kind, pa, ch = (int(joints["params"][j, i]) for i in range(3))
                c = _rotate(t64(joints["axis"][j, :3]).expand(E, 3), quat[:, pa]) * tau[:, j:j + 1]
                into = force if kind == 2 else torque
                for b, s in ((pa, -1.0), (ch, 1.0)):
                    if b != 0:
                        into[:, b] += s * c
            vel = torch.where(moves, (vel + force * inv_m * dt) * 0.999, vel)
            ang = torch.where(moves, (ang + inv_i * torque * dt) * 0.999, ang)
            pos = torch.where(moves, pos + vel * dt, pos)
            w = torch.cat([ang * dt * 0.5, torch.zeros_like(ang[..., :1])], -1)
            quat = torch.where(moves, _unit(quat + _qmul(w, quat)), quat)
            for _ in range(4):
                for n, c in enumerate(m["constraints"]):
                    _solve_joint(c, n, pos, quat, lam, inv_m, inv_i, com, dt, t64, turn)
            vel = torch.where(moves, (pos - pos0) / dt, vel)
            d = _qmul(quat, _conj(quat0))
            d = torch.where(d[..., 3:] < 0, -d, d)
            ang = torch.where(moves, 2.0 * d[..., :3] / dt, ang)
        q, qd = torch.zeros_like(tau), torch.zeros_like(tau)
        for j in range(J):
            kind, pa, ch = (int(joints["params"][j, i]) for i in range(3))
            axis = t64(joints["axis"][j, :3]).expand(E, 3)
            aw = _rotate(axis, quat[:, pa])
            if kind == 1:
                rel = _qmul(_conj(quat[:, pa]), quat[:, ch])
                q[:, j] = 2.0 * torch.atan2(_dot(rel[..., :3], axis)[:, 0], rel[..., 3])
                qd[:, j] = _dot(ang[:, ch] - ang[:, pa], aw)[:, 0]
            elif kind == 2:
                ra = _rotate(t64(joints["anchor_parent"][j, :3]).expand(E, 3), quat[:, pa])
                rb = _rotate(t64(joints["anchor_child"][j, :3]).expand(E, 3), quat[:, ch])
                q[:, j] = _dot(pos[:, ch] + rb - pos[:, pa] - ra, aw)[:, 0]
                va = vel[:, pa] + torch.linalg.cross(ang[:, pa], ra, dim=-1)
                vb = vel[:, ch] + torch.linalg.cross(ang[:, ch], rb, dim=-1)
                qd[:, j] = _dot(vb - va, aw)[:, 0]
        obs = torch.zeros(E, m["obs_dim"], dtype=torch.float64, device=dev)
        for s in m["sensors"]:
            kind, j, at = int(s["type_object"][0]), int(s["type_object"][1]), int(s["params"][3])
            obs[:, at] = q[:, j] if kind == 0 else qd[:, j]
    return obs


def _solve_joint(c, n, pos, quat, lam, inv_m, inv_i, com, dt, t64, turn):
    """One constraint of the scene's list on every environment (types: 2 point, 3 hinge axis,
    5 linear limit, 7 weld, 10 slider)."""
    E = pos.shape[0]
    a, b, kind = int(c["indices"][0]), int(c["indices"][1]), int(c["indices"][3]) & 0xFF
    if float(inv_m[a] + inv_m[b]) < 1e-8:
        return
    soft = float(c["anchor_a"][3]) / dt ** 2
    va, vb = t64(c["anchor_a"][:3]).expand(E, 3), t64(c["anchor_b"][:3]).expand(E, 3)
    third = t64(c["axis_target"]).expand(E, 4)

    def weight(r, dirn, body):
        rn = torch.linalg.cross(r, dirn, dim=-1)
        return inv_m[body] + _dot(rn * inv_i[body], rn)

    def push(body, imp, r, sign, mask):
        if float(inv_m[body]) > 0:
            imp = torch.where(mask, imp, torch.zeros_like(imp))
            before = quat[:, body].clone()
            pos[:, body] += sign * imp * inv_m[body]
            turn(body, torch.linalg.cross(r, imp, dim=-1), sign)
            quat[:, body] = torch.where(mask, quat[:, body], before)

    def align(target, both):  # relative orientation driven to target
        err = _qmul(_qmul(_conj(quat[:, a]), quat[:, b]), _conj(target))
        err = torch.where(err[..., 3:] < 0, -err, err)
        sh = err[..., :3].norm(dim=-1, keepdim=True)
        axis = _rotate(_unit(err[..., :3]), quat[:, a])
        w = _dot(axis * inv_i[b], axis) + (_dot(axis * inv_i[a], axis) if both else 0.0)
        on = (sh > 1e-6) & (w > 1e-8)
        imp = torch.where(on, 2.0 * torch.atan2(sh, err[..., 3:]) / (w + soft), torch.zeros_like(sh)) * axis
        for body, sign in ((a, 1.0), (b, -1.0)):
            if float(inv_m[body]) > 0 and (both or body == b):
                before = quat[:, body].clone()
                turn(body, imp, sign)
                quat[:, body] = torch.where(on, quat[:, body], before)

    if kind in (2, 7):
        ra, rb = _rotate(va, quat[:, a]), _rotate(vb, quat[:, b])
        diff = pos[:, a] + ra - pos[:, b] - rb
        err = diff.norm(dim=-1, keepdim=True)
        dirn, on = _unit(diff), err > 1e-6
        if kind == 2:
            dl = (-err - soft * lam[:, n:n + 1]) / (weight(ra, dirn, a) + weight(rb, dirn, b) + soft)
            ca, cb = (_rotate(com[x].expand(E, 3), quat[:, x]) for x in (a, b))
            push(a, dl * dirn, ra - ca, 1.0, on)
            push(b, dl * dirn, rb - cb, -1.0, on)
            lam[:, n:n + 1] += torch.where(on, dl, torch.zeros_like(dl))
        else:
            push(b, -err / (weight(rb, dirn, b) + soft) * dirn, rb, -1.0, on)
            align(third, False)
    elif kind == 3:
        cr = torch.linalg.cross(_rotate(va, quat[:, a]), _rotate(vb, quat[:, b]), dim=-1)
        s = cr.norm(dim=-1, keepdim=True)
        axis = _unit(cr)
        w = _dot(axis * inv_i[a], axis) + _dot(axis * inv_i[b], axis)
        imp = torch.where(s > 1e-6, -torch.asin(s.clamp(-1, 1)) / (w + soft), torch.zeros_like(s)) * axis
        for body, sign in ((a, 1.0), (b, -1.0)):
            if float(inv_m[body]) > 0:
                turn(body, sign * imp, 1.0)
    elif kind == 5:
        aw = _rotate(va, quat[:, a])
        rb = _rotate(vb, quat[:, b])
        d = _dot(pos[:, b] + rb - pos[:, a], aw)
        lo, hi = float(c["limits"][0]), float(c["limits"][1])
        off = torch.where(d < lo, lo - d, torch.where(d > hi, hi - d, torch.zeros_like(d)))
        dirn = torch.where(off > 0, aw, -aw)
        imp = off.abs() / (inv_m[a] + weight(rb, dirn, b) + soft) * dirn
        for body, sign in ((a, -1.0), (b, 1.0)):
            if float(inv_m[body]) > 0:
                pos[:, body] += sign * imp * inv_m[body]
    elif kind == 10:
        ra, rb = _rotate(va, quat[:, a]), _rotate(vb, quat[:, b])
        aw = _rotate(third[:, :3], quat[:, a])
        diff = pos[:, a] + ra - pos[:, b] - rb
        perp = diff - _dot(diff, aw) * aw
        err = perp.norm(dim=-1, keepdim=True)
        dirn = _unit(perp)
        imp = -err / (weight(ra, dirn, a) + weight(rb, dirn, b) + soft) * dirn
        push(a, imp, ra, 1.0, err > 1e-6)
        push(b, imp, rb, -1.0, err > 1e-6)
        align(t64(c["limits"]).expand(E, 4), True)


def _exact_collide(case, seed):
    where = "cuda" if case["where"] == "device" else "cpu"
    a, b = _collide_operands(case, seed, where)
    n = case["pairs"]
    out = {"point": torch.zeros(n, 3, dtype=torch.float64, device=where), "normal": torch.zeros(n, 3, dtype=torch.float64, device=where),
           "penetration": torch.zeros(n, dtype=torch.float64, device=where), "valid": torch.zeros(n, dtype=torch.int32, device=where),
           "local_a": torch.zeros(n, 4, dtype=torch.float64, device=where), "local_b": torch.zeros(n, 4, dtype=torch.float64, device=where)}
    kinds = a.view(torch.int32)[:, 0] * 4 + b.view(torch.int32)[:, 0]
    test = {(0, 0): _ss, (0, 1): _sc, (0, 2): _sb, (0, 3): _sp, (1, 1): _cc, (1, 3): _cp, (2, 3): _bp, (2, 2): _bb}
    for ka in range(4):
        for kb in range(4):
            swap = (ka, kb) not in test
            if swap and (kb, ka) not in test:
                continue
            at = (kinds == ka * 4 + kb).nonzero()[:, 0]
            x, y = a[at].double(), b[at].double()
            point, normal, pen, la, lb, ok = test[(kb, ka)](y, x) if swap else test[(ka, kb)](x, y)
            if swap:
                normal, la, lb = -normal, lb, la
            at, ok = at[ok], ok.nonzero()[:, 0]
            out["point"][at], out["normal"][at], out["penetration"][at] = point[ok], normal[ok], pen[ok, 0]
            out["local_a"][at, :3], out["local_b"][at, :3], out["valid"][at] = la[ok], lb[ok], 1
    # Host results come as numpy arrays, whatever holds them here.
    return {k: v.numpy() if where == "cpu" else v for k, v in out.items()}


def _pose(r):
    return r[:, 8:11], r[:, 12:16], r[:, 1:4]


def _axis(q, k):
    e = torch.zeros(q.shape[0], 3, dtype=q.dtype, device=q.device)
    e[:, k] = 1.0
    return _rotate(e, q)


def _round_pair(pa, ra, pb, rb, mid):
    """Two points with radii: contact along their difference; mid(normal, depth) places it."""
    d = pb - pa
    dist = d.norm(dim=-1, keepdim=True)
    up = torch.zeros_like(d)
    up[:, 2] = 1.0
    n = torch.where(dist > 1e-6, _unit(d), up)
    pen = ra + rb - dist
    return mid(n, pen), n, pen, n * ra, -n * rb, (pen > 0)[:, 0]


def _ss(a, b):
    pa, ra = a[:, 8:11], a[:, 1:2]
    return _round_pair(pa, ra, b[:, 8:11], b[:, 1:2], lambda n, pen: pa + n * (ra - 0.5 * pen))


def _sc(a, b):
    sp, sr, (cp, q, size) = a[:, 8:11], a[:, 1:2], _pose(b)
    cr, axis = size[:, :1], _axis(q, 2)
    near = cp + axis * torch.minimum(torch.maximum(_dot(sp - cp, axis), -size[:, 1:2]), size[:, 1:2])
    # The normal runs from the capsule to the sphere, scaled by each one's own radius.
    point, n, pen, lc, ls, ok = _round_pair(near, cr, sp, sr, lambda n, pen: near + n * (cr - 0.5 * pen))
    return point, n, pen, -ls, -lc, ok


def _sp(a, b):
    sp, sr, (pp, q, size) = a[:, 8:11], a[:, 1:2], _pose(b)
    n = _axis(q, 2)
    d = _dot(sp - pp, n) - size[:, :1]
    pen = sr - d
    return sp - n * (d + 0.5 * pen), n, pen, -n * sr, torch.zeros_like(n), (pen > 0)[:, 0]


def _sb(a, b):
    sp, sr, (pos, q, he) = a[:, 8:11], a[:, 1:2], _pose(b)
    local = _rotate(sp - pos, _conj(q))
    cl = torch.minimum(torch.maximum(local, -he), he)
    d = local - cl
    dist = d.norm(dim=-1, keepdim=True)
    far = torch.stack([he - local, he + local], -1).reshape(-1, 6)  # distance to +x, -x, +y, ... faces
    k = far.argmax(-1)
    face = torch.zeros_like(local)
    face[torch.arange(len(k), device=k.device), k // 2] = 1.0 - 2.0 * (k % 2).to(local.dtype)
    n = _rotate(torch.where(dist > 1e-6, _unit(d), face), q)
    pen = sr - dist
    return _rotate(cl, q) + pos + 0.5 * pen * n, n, pen, -n * sr, cl, (pen > 0)[:, 0]


def _cc(a, b):
    pa, qa, sa = _pose(a)
    pb, qb, sb = _pose(b)
    xa, xb = _axis(qa, 2), _axis(qb, 2)
    a1, b1 = pa - xa * sa[:, 1:2], pb - xb * sb[:, 1:2]
    d1, d2 = 2.0 * xa * sa[:, 1:2], 2.0 * xb * sb[:, 1:2]
    r = a1 - b1
    A, e, f, c, bb = _dot(d1, d1), _dot(d2, d2), _dot(d2, r), _dot(d1, r), _dot(d1, d2)
    s = ((bb * f - c * e) / (A * e - bb * bb)).clamp(0, 1)
    t = (bb * s + f) / e
    s = torch.where(t < 0, (-c / A).clamp(0, 1), torch.where(t > 1, ((bb - c) / A).clamp(0, 1), s))
    t = t.clamp(0, 1)
    p, w, ra, rb = a1 + d1 * s, b1 + d2 * t, sa[:, :1], sb[:, :1]
    return _round_pair(p, ra, w, rb, lambda n, pen: 0.5 * (p + n * ra + w - n * rb))


def _cp(a, b):
    (cp, qc, size), (pp, q, _) = _pose(a), _pose(b)
    n, axis = _axis(q, 2), _axis(qc, 2)
    ends = [cp - axis * size[:, 1:2], cp + axis * size[:, 1:2]]
    d = [_dot(x - pp, n) - size[:, :1] for x in ends]
    first = d[0] < d[1]
    depth, deep = torch.where(first, d[0], d[1]), torch.where(first, ends[0], ends[1])
    return deep - n * (0.5 * depth + size[:, :1]), n, -depth, -n * size[:, :1], torch.zeros_like(n), (depth < 0)[:, 0]


def _bp(a, b):
    (pos, q, he), (pp, qp, _) = _pose(a), _pose(b)
    n = _axis(qp, 2)
    corners = torch.stack([he * torch.tensor([1.0 if k >> i & 1 else -1.0 for i in range(3)], dtype=he.dtype, device=he.device)
                           for k in range(8)], 1)
    world = _rotate(corners, q[:, None].expand(-1, 8, 4)) + pos[:, None]
    d = _dot(world - pp[:, None], n[:, None].expand(-1, 8, 3))[..., 0]
    depth, k = d.min(1, keepdim=True)
    at = k[:, :, None].expand(-1, 1, 3)
    return world.gather(1, at)[:, 0], n, -depth, corners.gather(1, at)[:, 0], torch.zeros_like(n), (depth < 0)[:, 0]


def _bb(a, b):
    (pa, qa, ha), (pb, qb, hb) = _pose(a), _pose(b)
    xa, xb = [_axis(qa, k) for k in range(3)], [_axis(qb, k) for k in range(3)]
    d = pb - pa
    best = torch.full_like(d[:, :1], math.inf)
    normal = torch.zeros_like(d)
    for axis in xa + xb + [torch.linalg.cross(x, y, dim=-1) for x in xa for y in xb]:
        size = axis.norm(dim=-1, keepdim=True)
        axis = _unit(axis)
        reach = sum(ha[:, k:k + 1] * _dot(axis, xa[k]).abs() + hb[:, k:k + 1] * _dot(axis, xb[k]).abs() for k in range(3))
        over = torch.where(size < 1e-6, torch.full_like(best, math.inf), reach - _dot(d, axis).abs())
        closer = over < best
        best, normal = torch.where(closer, over, best), torch.where(closer, axis, normal)
    normal = torch.where(_dot(normal, d) < 0, -normal, normal)
    return pa + 0.5 * d, normal, best, torch.zeros_like(d), torch.zeros_like(d), (best >= 0)[:, 0]
