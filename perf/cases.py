"""Performance cases of the batched stepping engine.

What a program that uses the engine has it do, through the entry points such
a program calls: one vector step of an environment loop (resets, inputs, the
masked b3_step of every world) on worlds resident on the GPU, the PufferLib
hover environment's step, and the step of worlds the caller keeps in its own
device memory.  The five world families and their capacities, step sizes and
batch sizes are puffysics_amd.scenes.SCENES (the workloads bench.py times);
the other batch sizes and the optional steps (gravity law, articulated
contacts) are those of the tests.

A pass is one vector step: the state moves on from pass to pass, as in a
rollout.  Its outputs are the state the step leaves behind: the world counts
(contacts found and dropped, overflow flags), every body's record and, where
the family has joints, every joint's record, as views of the engine's own
device memory; for the hover environment also its observations, rewards and
terminals.  Contact records past a world's contact count hold whatever was
last there and are not returned; the impulses of the live ones decide the
next pass.

The step's contract is the reference's fp32 result bit for bit (the solver
runs a fixed number of Gauss-Seidel sweeps in a fixed order, so another
order or precision is another result), hence tolerance "exact".
"""
import ctypes as C

import numpy as np
import torch

from puffysics_amd import _native, scenes
from puffysics_amd.b3types import B3Batch, world_ctype
from puffysics_amd.engine import B3_ENGINE_ART_CONTACTS, B3Engine, device_tensor
from puffysics_amd.hover import HoverEnvs

HOVER, STACK, CHAIN, BIN, ARM = 1, 2, 3, 4, 5

#: Vector steps before the first pass: the stacks stand, the bin's bodies
#: have landed, the arm's resets run at their steady rate.
SETTLE = {HOVER: 500, STACK: 500, CHAIN: 500, BIN: 1000, ARM: 500}
#: Masks drawn ahead by the policy (the arm: 2% resets, 90% stepped).
MASKS = 32
#: The hover environment's steps before the first pass, and how many of them
#: hold one action.
ENV_STEPS, ENV_HOLD = 96, 16


def listed():
    return [
        # the hover task's vector step at a small and at PufferLib's usual
        # number of envs: launches and latency are all of it
        {"name": "env_64", "kind": "env", "scene": HOVER, "worlds": 64},
        {"name": "env_4096", "kind": "env", "scene": HOVER, "worlds": 4096},
        # the benchmark's families at its batch sizes: one body over the
        # ground, box stacks, hinge chains, a bin of mixed bodies
        {"name": "hover_4096", "kind": "step", "scene": HOVER, "worlds": 4096},
        {"name": "stack_4096", "kind": "step", "scene": STACK, "worlds": 4096},
        {"name": "chain_4096", "kind": "step", "scene": CHAIN, "worlds": 4096},
        {"name": "bin_4096", "kind": "step", "scene": BIN, "worlds": 4096},
        # a hinged arm with free bodies, masked resets and steps: a small
        # evaluation batch (resets fused into the step), a middle batch of
        # odd size, and the scale benchmark
        {"name": "arm_300", "kind": "fused", "scene": ARM, "worlds": 300},
        {"name": "arm_17000", "kind": "step", "scene": ARM, "worlds": 17000},
        {"name": "arm_65536", "kind": "step", "scene": ARM, "worlds": 65536},
        # a serving loop that may not allocate: the caller's own worlds
        {"name": "arm_worlds_2000", "kind": "worlds", "scene": ARM, "worlds": 2000},
        # the optional steps: pairwise gravity, articulated contacts
        {"name": "arm_gravity_1000", "kind": "gravity", "scene": ARM, "worlds": 1000},
        {"name": "arm_art_1000", "kind": "art", "scene": ARM, "worlds": 1000},
    ]


#: Batch sizes of drawn cases: (kind, scene, fewest, most, weight).
RANGES = [
    ("env", HOVER, 16, 16384, 2),
    ("step", HOVER, 64, 65536, 2),
    ("step", STACK, 64, 16384, 2),
    ("step", CHAIN, 64, 16384, 2),
    ("step", BIN, 64, 8192, 2),
    ("step", ARM, 64, 40000, 3),
    ("fused", ARM, 64, 16384, 1),
    ("worlds", ARM, 64, 2000, 1),
    ("gravity", ARM, 64, 4096, 1),
    ("art", ARM, 64, 1000, 1),
]


def draw(rng):
    kind, scene, lo, hi, _ = rng.choices(RANGES, weights=[r[4] for r in RANGES])[0]
    n = int(round(lo * (hi / lo) ** rng.random()))
    return {"kind": kind, "scene": scene, "worlds": max(lo, min(hi, n))}


class State:
    pass


class Outputs(dict):
    """A pass's outputs by name.  Views of device memory that an engine or an
    environment owns hold it (`owner`): the memory goes with its owner."""


def _out_tiles(tiles, sig, scene, owner):
    """The returned views of [tiles, words, 64] int32 world tiles."""
    w = world_ctype(sig)
    bo, so, jo = w.bodies.offset // 4, w.shapes.offset // 4, w.joints.offset // 4
    je = C.sizeof(w) // 4
    out = Outputs(counts=tiles[:, w.body_count.offset // 4:bo, :], bodies=tiles[:, bo:so, :].view(torch.float32))
    out.owner = owner
    if scene in (CHAIN, ARM):
        out["joints"] = tiles[:, jo:je, :].view(torch.float32)
    return out


def _settled(scene, n, seed):
    """An engine of `n` worlds of the scene after its settling steps."""
    sc = scenes.SCENES[scene]
    worlds = scenes.build(scene, n, seed=seed)
    eng = B3Engine(worlds, sc.sig)            # its snapshots are the initial worlds
    reset = torch.zeros(n, dtype=torch.uint8, device="cuda")
    step = torch.zeros(n, dtype=torch.uint8, device="cuda")
    for t in range(SETTLE[scene]):
        if scene == ARM:
            eng.scene_masks(scene, seed, t, reset, step)
            eng.restore(reset)
            eng.scene_inputs(scene, seed, t, step)
            eng.step(sc.dt, sc.substeps, step)
        else:
            eng.scene_inputs(scene, seed, t)
            eng.step(sc.dt, sc.substeps)
    return eng


def prepare(case, seed):
    s = State()
    s.kind, s.scene, n = case["kind"], case["scene"], case["worlds"]
    s.sc = scenes.SCENES[s.scene]
    s.seed, s.t, s.n = seed, SETTLE[s.scene], n
    if s.kind == "env":
        s.env = HoverEnvs(n, seed=seed & 0x7fffffff)
        s.env.reset()
        acts = _env_actions(n, seed)
        for i in range(ENV_STEPS):
            if i % ENV_HOLD == 0:
                s.env.actions.copy_(torch.from_numpy(acts[i // ENV_HOLD]))
            s.env.step()
        s.env.actions.copy_(torch.from_numpy(acts[-1]))    # the policy's answer to the last observations
        ptr, words = C.c_void_p(), C.c_size_t()
        code = _native.engine_lib().b3_engine_device_view(s.env.engine_handle(), C.byref(ptr), C.byref(words))
        assert code == 0
        s.out = _out_tiles(device_tensor(ptr.value, ((n + 63) // 64, words.value, 64)), s.sc.sig, s.scene, s.env)
        s.out.update(observations=s.env.observations, rewards=s.env.rewards, terminals=s.env.terminals)
        return s
    s.eng = _settled(s.scene, n, seed)
    s.reset = s.step = None
    if s.scene == ARM:
        s.reset = torch.zeros((MASKS, n), dtype=torch.uint8, device="cuda")
        s.step = torch.zeros((MASKS, n), dtype=torch.uint8, device="cuda")
        for k in range(MASKS):
            s.eng.scene_masks(s.scene, seed, s.t + k, s.reset[k], s.step[k])
    if s.kind == "art":
        s.eng.set_options(B3_ENGINE_ART_CONTACTS)
    if s.kind == "worlds":
        worlds = s.eng.download()
        s.eng.close()
        s.eng = None
        s.dev = torch.from_numpy(worlds.view(np.uint8).reshape(n, -1)).cuda()
        s.batch = B3Batch(s.dev.data_ptr(), worlds.dtype.itemsize, 0, n)
        w, words = world_ctype(s.sc.sig), s.dev.view(torch.int32)
        bo, so, jo = w.bodies.offset // 4, w.shapes.offset // 4, w.joints.offset // 4
        s.out = {"counts": words[:, w.body_count.offset // 4:bo], "bodies": words[:, bo:so].view(torch.float32),
                 "joints": words[:, jo:].view(torch.float32)}
        return s
    s.out = _out_tiles(s.eng.tiles(), s.sc.sig, s.scene, s.eng)
    return s


def run(s):
    sc = s.sc
    if s.kind == "env":
        s.env.step()
        return s.out
    k = (s.t - SETTLE[s.scene]) % MASKS
    if s.kind == "worlds":
        code = _native.engine_lib().b3_batch_step_worlds_gpu(s.batch, sc.sig, sc.dt, sc.substeps, s.step[k].data_ptr(),
                                                             torch.cuda.current_stream().cuda_stream)
        if code != 0:
            raise RuntimeError("b3_batch_step_worlds_gpu failed with %d" % code)
        s.t += 1
        return s.out
    reset = step = None
    if s.step is not None:
        reset, step = s.reset[k], s.step[k]
    if s.kind == "fused":
        s.eng.scene_inputs(s.scene, s.seed, s.t, step)
        s.eng.step(sc.dt, sc.substeps, step, reset)
    else:
        if reset is not None:
            s.eng.restore(reset)
        s.eng.scene_inputs(s.scene, s.seed, s.t, step)
        if s.kind == "gravity":
            s.eng.step_gravity(sc.dt, sc.substeps, 2.0, 0.1, step_mask=step)
        else:
            s.eng.step(sc.dt, sc.substeps, step)
    s.t += 1
    return s.out


#: Per world of a family: dynamic bodies, static bodies, shapes, joints, mean
#: live contacts of the settled worlds, and the step's fp32 operations
#: (counted on the CPU oracle over the settled worlds, tests/golden).
FAMILY = {
    HOVER: (1, 1, 2, 0, 0.3, 2.5e3),
    STACK: (5, 1, 6, 0, 5.6, 5.2e4),
    CHAIN: (8, 1, 8, 8, 0.0, 2.47e5),
    BIN: (32, 1, 37, 0, 40.9, 2.32e5),
    ARM: (16, 1, 17, 4, 12.3, 1.44e5),
}


def work(case):
    """A stepped world's persistent state once through memory: a dynamic body
    212 bytes (76 read, 64 written, 24 of force and torque cleared, 48 of
    constants), a static one 36, a shape 80, a live contact 136 (its warm
    cache read and written), a joint 192, the world 58; a reset world its
    bodies and joints read and written."""
    n = case["worlds"]
    if case["kind"] == "env":      # one free sphere; observation, action, reward, terminal
        return {"bytes": n * (212 + 80 + 58 + 24), "flops": n * 6.0e2}
    dyn, static, shapes, joints, contacts, flops = FAMILY[case["scene"]]
    world = 212 * dyn + 36 * static + 80 * shapes + 192 * joints + 136 * contacts + 58
    stepped, resets = (0.9, 0.02) if case["scene"] == ARM else (1.0, 0.0)
    if case["kind"] in ("worlds", "gravity", "art"):
        resets = 0.0 if case["kind"] == "worlds" else resets
    if case["kind"] == "gravity":
        flops += 4 * 17 * 16 / 2 * 30
    return {"bytes": n * world * (stepped + 2 * resets), "flops": n * stepped * flops}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """The hover environment in 64 bits: a free body under gravity and its
    thrust, in closed form per substep.  The other families have no value in
    64 bits to compare with: their inputs are worlds settled over hundreds of
    steps by the code itself, and a contact or joint solve is cut off after a
    fixed number of sweeps whose order is the result; it is held to the
    bits."""
    if case["kind"] != "env":
        return None
    n = case["worlds"]
    env_seed = seed & 0x7fffffff
    target, thrust, dt, subs, horizon, gravity = 2.0, 10.0, 1.0 / 60.0, 4, 256, -10.0
    with np.errstate(over="ignore"):
        rng = np.uint32(env_seed) + np.arange(n, dtype=np.uint32) * np.uint32(747796405)

        def lcg(r):
            return r * np.uint32(1664525) + np.uint32(1013904223)

        def start(r):
            return target + (r >> np.uint32(8)).astype(np.float64) / 16777216.0 - 0.5

        rng = lcg(lcg(rng))                       # create draws once, reset again
        y, vy, tick = start(rng), np.zeros(n), np.zeros(n, np.int64)
        acts = _env_actions(n, seed)
        h = dt / subs
        for i in range(ENV_STEPS + 1):
            a = acts[i // ENV_HOLD] if i < ENV_STEPS else acts[-1]
            level = np.where(a >= 1.5, 2.0, np.where(a >= 0.5, 1.0, 0.0))
            for _ in range(subs):
                vy = vy + h * (gravity + level * thrust)
                y = y + h * vy
            tick += 1
            e = np.abs(y - target) + 0.1 * np.abs(vy)
            reward = 1.0 - np.minimum(e, 2.0)
            done = (np.abs(y - target) > 3.0) | (tick >= horizon)
            rng = np.where(done, lcg(rng), rng)
            y, vy, tick = np.where(done, start(rng), y), np.where(done, 0.0, vy), np.where(done, 0, tick)
    obs = np.stack([y - target, vy, tick / horizon], axis=1)
    return {"counts": None, "bodies": None, "observations": torch.from_numpy(obs),
            "rewards": torch.from_numpy(reward), "terminals": torch.from_numpy(done.astype(np.float64))}


def _env_actions(n, seed):
    """The policy's actions, one row per hold, the last for the timed pass."""
    rows = ENV_STEPS // ENV_HOLD + 1
    return np.random.default_rng([seed, n]).uniform(0.0, 2.0, (rows, n)).astype(np.float32)
