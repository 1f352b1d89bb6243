"""The work that a user of this framework has it do, as measurable cases.

A case is one pass through the public entry points of nans_projekat_amd.runtime:
  pairs   Context.narrowphase on device-resident pairs (GJK and EPA contact query);
  plain   Context.set_state, step_plain, download: one scene, the drop-in step;
  batch   Context.set_state, step_batched, download: an episode of many worlds;
  grad    Context.set_state, rollout, adjoint: one gradient of a rollout.
Stepping cases start every pass from the state that prepare() uploaded, as an
episode or an optimiser's rollout does, so that every pass is the same work.
"""
import dataclasses
import math

import numpy as np

from nans_projekat_amd import runtime
from nans_projekat_amd import scenes as S

# Floating-point operations of a body per step (RK4, Model rebuild, cull, GJK, EPA,
# impulse iterations), from the CPU oracle's event counts on scenes of these kinds
# (mul, add, sub, div and sqrt count 1), and of a random narrowphase pair.
FLOPS_STACK = 7000.0
FLOPS_LAYER = 3600.0
FLOPS_DROP = 2500.0
FLOPS_PAIR = 2070.0
# State of a body: read position, velocity, angular velocity, angles, scale, mass, moment of
# inertia, force and torque; write all but scale, mass and moment of inertia.
BYTES_BODY = 92 + 72
# A pair: two shapes of 44 bytes in, flags, status, normal, depth and both points out.
BYTES_PAIR = 144
# The state fields that set_state takes and download returns.
STATE = ("pos", "vel", "angvel", "angles", "force", "torque")


def listed():
    return [
        # a contact query from a user's own loop: a few hundred pairs, where the call's latency counts
        dict(name="pairs_777", kind="pairs", n=777, islands=0),
        # the candidates of a mid-sized scene, not a multiple of any tile
        dict(name="pairs_30011", kind="pairs", n=30011, islands=0),
        # the same query in the binary64-islands mode
        dict(name="pairs_islands_200k", kind="pairs", n=200_000, islands=1),
        # the narrowphase benchmark's size
        dict(name="pairs_1m", kind="pairs", n=1_000_000, islands=0),
        # a game loop: 28 bodies, one step and one read-back per frame
        dict(name="frames_stack28", kind="plain", scene="stack28", bodies=28, frames=40, per_frame=1),
        # one mid-sized scene, ten steps per read-back
        dict(name="scene_181", kind="plain", scene="stack", bodies=181, frames=4, per_frame=10),
        # the large world, from the drop well into the landing
        dict(name="large_8192", kind="plain", scene="drop", bodies=8192, frames=1, per_frame=240),
        # a handful of small worlds (a planner's samples): fewer than the chip has compute units
        dict(name="batch_48", kind="batch", worlds=48, lo=8, hi=64, steps=30, mode="euler", warm=0),
        # a few hundred uneven worlds with the opt-in quaternion orientation and warm start
        dict(name="batch_601_modes", kind="batch", worlds=601, lo=8, hi=256, steps=30, mode="quaternion", warm=1),
        # the batched benchmark's 4096 uneven worlds, half a second of simulated time
        dict(name="batch_4096", kind="batch", worlds=4096, lo=8, hi=256, steps=60, mode="euler", warm=0),
        # one gradient over a few small worlds, segments of odd length
        dict(name="grad_24", kind="grad", worlds=24, gx=3, gz=3, steps=50, every=7),
        # the differentiable benchmark: 1024 worlds of 16 cubes, 240 steps, checkpoints every 16
        dict(name="grad_1024", kind="grad", worlds=1024, gx=4, gz=4, steps=240, every=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("pairs", "pairs", "plain", "plain", "batch", "batch", "grad"))
    if kind == "pairs":
        return dict(kind=kind, n=_log(rng, 300, 1_000_000), islands=rng.choice((0, 0, 1)))
    if kind == "plain":
        if rng.random() < 0.35:
            return dict(kind=kind, scene="drop", bodies=_log(rng, 1100, 8192), frames=1, per_frame=rng.randint(60, 240))
        return dict(kind=kind, scene="stack", bodies=_log(rng, 8, 512), frames=rng.randint(1, 20),
                    per_frame=rng.randint(1, 12))
    if kind == "batch":
        lo = _log(rng, 5, 24)
        return dict(kind=kind, worlds=_log(rng, 2, 3000), lo=lo, hi=lo + _log(rng, 2, 230), steps=rng.randint(5, 60),
                    mode=rng.choice(("euler", "euler", "quaternion")), warm=rng.choice((0, 0, 1)))
    return dict(kind=kind, worlds=_log(rng, 4, 1024), gx=rng.randint(2, 5), gz=rng.randint(2, 4),
                steps=rng.randint(10, 160), every=rng.randint(1, 24))


# ---------------------------------------------------------------------- scenes
def _sizes(case):
    """Body counts of a batch's worlds: the quantiles of the log-uniform distribution over [lo, hi]."""
    w = case["worlds"]
    u = (np.arange(w) + 0.5) / w
    n = np.floor(np.exp(np.log(case["lo"]) + u * (np.log(case["hi"] + 1) - np.log(case["lo"])))).astype(np.int64)
    return np.clip(n, case["lo"], case["hi"])


def _stacks(sizes, r):
    """Worlds of jittered stacks of unit cubes on the ground, one to four spheres thrown at each."""
    nw = len(sizes)
    nsph = r.integers(1, 5, nw)
    nb = sizes - nsph
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    w = np.repeat(np.arange(nw), sizes)
    i = np.arange(offsets[-1]) - offsets[w]
    box = i < nb[w]
    side = np.maximum(1, np.rint(np.cbrt(nb)).astype(np.int64))
    layer, rem = i // (side[w] ** 2), i % (side[w] ** 2)
    off = (side[w] - 1) / 2.0
    pos = np.stack([1.2 + rem % side[w] - off, 0.5 + layer, 1.0 + rem // side[w] - off], axis=1)
    pos += r.uniform(-0.01, 0.01, pos.shape)
    n = len(w)
    centre = np.stack([np.full(nw, 1.2), 0.5 + ((nb - 1) // side ** 2) / 2.0, np.ones(nw)], axis=1)[w]
    az, rad, h = r.uniform(0, 2 * math.pi, n), r.uniform(6, 10, n) + side[w] / 2.0, r.uniform(0.5, 3, n)
    sph = np.stack([centre[:, 0] + rad * np.cos(az), h, centre[:, 2] + rad * np.sin(az)], axis=1)
    d = centre - sph
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    vel = np.where(box[:, None], 0.0, d * r.uniform(5, 25, n)[:, None])
    mass = np.where(box, 1.0, 2.0)
    moi = np.where(box, 1.0 / 6.0, 0.4 * 2.0 * 0.25)
    scale = np.where(box[:, None], 1.0, 0.5) * np.ones((1, 3))
    return _scene(np.where(box[:, None], pos, sph), vel, scale, mass, moi, np.where(box, S.BOX, S.SPHERE), offsets, nb)


def _layers(worlds, gx, gz, r):
    """Worlds of one layer of gx * gz cubes with their own masses, friction, restitution and velocities."""
    n = gx * gz
    g = np.array([(1.2 + 1.05 * (a - (gx - 1) / 2), 0.5, 1.0 + 1.05 * (b - (gz - 1) / 2)) for a in range(gx)
                  for b in range(gz)])
    pos = np.tile(g, (worlds, 1)) + r.uniform(-0.01, 0.01, (worlds * n, 3))
    mass = r.uniform(0.5, 2.0, worlds * n)
    sc = _scene(pos, r.normal(size=pos.shape), np.ones_like(pos), mass, mass / 6.0, np.full(worlds * n, S.BOX),
                (np.arange(worlds + 1) * n).astype(np.int32), np.full(worlds, n))
    sc.world_friction = r.uniform(0.2, 0.9, worlds).astype(np.float32)
    sc.world_restitution = r.uniform(0.0, 0.5, worlds).astype(np.float32)
    return sc


def _scene(pos, vel, scale, mass, moi, kind, offsets, nb):
    f = lambda a: np.ascontiguousarray(a, dtype=np.float32)
    z = lambda: np.zeros((len(pos), 3), np.float32)
    params = dataclasses.replace(S.StepParams(), solver_iterations=10, restitution=0.2, friction=0.5, dt=1.0 / 120.0)
    return S.Scene(f(pos), f(vel), z(), z(), z(), z(), f(scale), f(mass), f(moi), kind.astype(np.int32), offsets,
                   np.asarray(nb, np.int32), params, 0)


def _scene_of(case, seed):
    r = np.random.default_rng([seed, 7])
    if case["kind"] == "batch":
        return _stacks(r.permutation(_sizes(case)), r)
    if case["kind"] == "grad":
        return _layers(case["worlds"], case["gx"], case["gz"], r)
    if case["scene"] == "stack28":
        return S.config1(seed=seed)
    if case["scene"] == "stack":
        return _stacks(np.array([case["bodies"]]), r)
    # the jittered grid of boxes dropped from y >= 1: eight layers, the last one cut to the body count
    side = max(1, math.ceil(math.sqrt(case["bodies"] / 8)))
    sc = S.config5(seed=seed, nx=side, ny=8, nz=math.ceil(case["bodies"] / (8 * side)))
    m = case["bodies"]
    cut = lambda a: a[:m].copy()
    return dataclasses.replace(sc, **{k: cut(getattr(sc, k)) for k in STATE + ("scale", "mass", "moi", "kind")},
                               offsets=np.array([0, m], np.int32), nboxes=np.array([m], np.int32))


# ---------------------------------------------------------------------- what a program has, and does
def prepare(case, seed):
    if case["kind"] == "pairs":
        ctx = runtime.Context(fp64_islands=case["islands"])
        pairs = ctx.upload_pairs(S.config2_pairs(case["n"], seed=seed))
        return dict(case=case, ctx=ctx, pairs=pairs, out=ctx.alloc_narrow_out(case["n"]))
    scene = _scene_of(case, seed)
    ctx = runtime.Context(scene.params)
    ctx.upload(scene)
    state = dict(case=case, ctx=ctx, scene=scene)
    if case["kind"] == "batch":
        ctx.set_orientation_mode(case["mode"])
        ctx.set_warm_start(bool(case["warm"]))
    elif case["kind"] == "grad":
        # dL/d(final positions) of a mean squared distance to a target
        r = np.random.default_rng([seed, 8])
        state["dl_pos"] = (r.normal(size=scene.pos.shape) * (2.0 / len(scene.pos))).astype(np.float32)
    return state


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["kind"] == "pairs":
        return ctx.narrowphase(state["pairs"], state["out"])
    ctx.set_state(state["scene"])
    if case["kind"] == "grad":
        ctx.rollout(case["steps"], case["every"])
        return ctx.adjoint(dl_pos=state["dl_pos"])
    if case["kind"] == "batch":
        ctx.step_batched(case["steps"])
        return ctx.download()
    for _ in range(case["frames"]):
        ctx.step_plain(case["per_frame"])
        out = ctx.download()
    return out


def work(case):
    if case["kind"] == "pairs":
        return {"bytes": BYTES_PAIR * case["n"], "flops": FLOPS_PAIR * case["n"]}
    if case["kind"] == "plain":
        per = FLOPS_DROP if case["scene"] == "drop" else FLOPS_STACK
        return {"bytes": BYTES_BODY * case["bodies"], "flops": per * case["bodies"] * case["frames"] * case["per_frame"]}
    if case["kind"] == "batch":
        n = int(_sizes(case).sum())
        return {"bytes": BYTES_BODY * n, "flops": FLOPS_STACK * n * case["steps"]}
    # the rollout, and a reverse pass that replays each step and runs its adjoint
    n = case["worlds"] * case["gx"] * case["gz"]
    return {"bytes": 2 * BYTES_BODY * n, "flops": 3 * FLOPS_LAYER * n * case["steps"]}


def exact(case, seed):
    """No value: which pairs touch, with which face, normal and points, is what the engine's own
    binary32 decision rules say (its GJK misses a quarter of random overlaps that separating axes
    find), not what geometry in 64 bits says, and a step's bodies follow from all its contacts.
    Outputs are comparable bit for bit instead."""
    return None
