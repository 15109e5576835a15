"""The work that programs built on this framework have it do, as measurable
cases: fresh small worlds, the frame loop of one world, single large worlds,
batches of uneven worlds and the serving loop, over both solver families, both
key widths, boxes, spheres and voxel bodies.

A case is a dict of plain values; `prepare` makes what a program has in hand
before the call (bodies drawn from the seed, and the world, batch or server it
keeps), `run` is one call sequence through the public entry points and returns
the bodies it reads back.

The long-lived worlds (frames, pile, gas, batch, voxel) go on from pass to
pass, as they do in a program; fresh worlds and served requests start anew in
every pass.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "beat-box_amd"))

import beatbox  # noqa: E402
import scenes  # noqa: E402

# Sleeping is on by default.  The frame loops switch it off: a scene this
# small comes to rest within a second of simulated time, and a world that has
# fallen asleep no longer steps its solver.
AWAKE = scenes.SIM_DEFAULT_FLAGS & ~scenes.SIM_SLEEPING_ENABLED
SOLVERS = {"pgs_soft": scenes.SOLVER_PGS_SOFT, "pgs": scenes.SOLVER_PGS, "avbd": scenes.SOLVER_AVBD}


def listed():
    return [
        # a request for a fresh small world stepped a few frames and read back
        # (planning, a unit of a larger job): launches and copies count
        dict(name="fresh_49", kind="fresh", scene="boxes", bodies=49, solver="pgs_soft", bits=30, steps=8),
        # the same call at an odd size near the top of its range, mixed shapes
        dict(name="fresh_1501", kind="fresh", scene="pile", bodies=1501, solver="avbd", bits=63, steps=8),
        # the reference application's frame: one step, counters and poses read
        # back; its tower scene (27 bodies) under AVBD
        dict(name="frame_towers_27", kind="frames", scene="towers", side=0, solver="avbd", iterations=5, frames=1),
        # the same frame with 1,000 cubes and the ground, colour-sweep PGS
        dict(name="frame_cubes_1001", kind="frames", scene="cubes", side=10, solver="pgs_soft", iterations=8, frames=1),
        # one large serving-size pile of boxes and spheres
        dict(name="pile_20000", kind="pile", bodies=20000, steps=40),
        # the largest pile configuration
        dict(name="pile_100000", kind="pile", bodies=100_000, steps=20),
        # broad-phase stress: a million spheres in flight
        dict(name="gas_1000000", kind="gas", bodies=1_000_000, steps=80),
        # 4,096 uneven worlds in one batch, the headline configuration
        dict(name="batch_4096", kind="batch", worlds=4096, lo=16, hi=2048, solver="pgs_soft", steps=32),
        # batched worlds on the per-island serial path (plain PGS)
        dict(name="island_513", kind="batch", worlds=513, lo=16, hi=2048, solver="pgs", steps=16),
        # concave voxel bodies mixed with boxes and spheres, AVBD
        dict(name="voxel_64", kind="voxel", worlds=64, bodies=200, steps=120),
        # requests of 64 to 20,000 bodies served to completion
        dict(name="serve_64", kind="serve", requests=64, lo=64, hi=20000, steps_lo=30, steps_hi=90),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fresh", "frames", "pile", "gas", "batch", "batch", "voxel", "serve"])
    if kind == "fresh":
        bits = rng.choice([30, 63])
        return dict(kind=kind, scene=rng.choice(["boxes", "pile"]), bodies=_log_int(rng, 9, 1000 if bits == 30 else 2048),
                    solver=rng.choice(["pgs_soft", "avbd"]), bits=bits, steps=rng.randint(4, 16))
    if kind == "frames":
        return dict(kind=kind, scene="cubes", side=rng.randint(2, 10), solver=rng.choice(["pgs_soft", "avbd"]),
                    iterations=rng.randint(4, 12), frames=rng.randint(1, 4))
    if kind == "pile":
        return dict(kind=kind, bodies=_log_int(rng, 1500, 100_000), steps=rng.randint(10, 20))
    if kind == "gas":
        return dict(kind=kind, bodies=_log_int(rng, 9000, 1_000_000), steps=rng.randint(20, 80))
    if kind == "batch":
        lo = _log_int(rng, 8, 128)
        return dict(kind=kind, worlds=_log_int(rng, 16, 1500), lo=lo, hi=_log_int(rng, 2 * lo, 2048),
                    solver=rng.choice(["pgs_soft", "pgs_soft", "pgs"]), steps=rng.randint(6, 16))
    if kind == "voxel":
        return dict(kind=kind, worlds=rng.randint(3, 64), bodies=_log_int(rng, 20, 200), steps=rng.randint(20, 100))
    return dict(kind="serve", requests=rng.randint(8, 48), lo=64, hi=_log_int(rng, 500, 20000), steps_lo=20,
                steps_hi=rng.randint(30, 80))


def _desc(solver, iterations=8, bits=63, flags=scenes.SIM_DEFAULT_FLAGS):
    if solver == "pgs":  # plain PGS runs on the per-island path
        flags &= ~scenes.SIM_USE_GRAPH_COLORING
    return beatbox.WorldDesc.make(**scenes.world_desc(
        solver=SOLVERS[solver], iterations=iterations, flags=flags, morton_bits=bits,
        quirks=scenes.QUIRKS_PARITY if bits == 30 else 0))


def _spread(n, lo, hi, rng):
    """n whole numbers spread evenly over log [lo, hi], in random order: every
    seed has the same sizes, so the same amount of work."""
    q = (np.arange(n) + 0.5) / n
    v = np.rint(np.exp(math.log(lo) + q * (math.log(hi) - math.log(lo)))).astype(np.int64)
    return rng.permutation(v)


def _stack_world(n, half, pyramid):
    """The batched configuration's world: a planar box pyramid or a tower of
    4 x 4 layers, n boxes on their own ground."""
    bodies = np.zeros(n + 1, scenes.BODY_DESC)
    scenes._ground(bodies[0])
    pos = np.zeros((n, 3))
    if pyramid:
        rows = int(math.ceil((math.sqrt(8 * n + 1) - 1) / 2))
        count = np.arange(rows, 0, -1)
        r = np.repeat(np.arange(rows), count)[:n]
        c = np.arange(n) - (np.cumsum(count) - count)[r]
        pos[:, 0] = (c - (count[r] - 1) / 2.0) * 2.0 * half * 1.04
        pos[:, 1] = half * 1.002 + r * 2.0 * half * 1.002
    else:
        layer, cell = np.divmod(np.arange(n), 16)
        cx, cz = np.divmod(cell, 4)
        pos[:, 0] = (cx - 1.5) * 2.0 * half * 1.03
        pos[:, 1] = half * 1.002 + layer * 2.0 * half * 1.002
        pos[:, 2] = (cz - 1.5) * 2.0 * half * 1.03
    b = bodies[1:]
    b["shape"] = scenes.SHAPE_BOX
    b["flags"] = scenes.BODY_DYNAMIC | scenes.BODY_GRAVITY
    b["position"] = pos
    b["rotation"] = (0.0, 0.0, 0.0, 1.0)
    b["minimum"] = -half
    b["maximum"] = half
    b["mass"] = (2 * half) ** 3
    b["friction"] = 0.5
    return bodies


class _Stepped:
    """A batch its program keeps, and the device buffer its poses go to."""

    def __init__(self, batch, counts, warm, tune):
        self.batch, self.counts = batch, counts
        batch.step(warm, use_graph=True)
        batch.sync(allow_overflow=True)
        if tune:
            batch.autotune(2)
        self.poses = torch.zeros(sum(counts), 12, dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
        at = self.poses.data_ptr() + 48 * np.concatenate([[0], np.cumsum(counts)[:-1]])
        self.targets = [(w, int(n), int(p)) for w, (n, p) in enumerate(zip(counts, at))]


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "fresh":
        n = case["bodies"]
        if case["scene"] == "boxes":
            bodies = scenes.random_boxes(seed, n - 1, extent=max(2.0, 0.6 * (n - 1) ** (1 / 3)), y0=0.55,
                                         y1=4.0 + 0.01 * n)
        else:
            bodies = scenes.serving_pile(seed, n - 1)
        return dict(case=case, desc=_desc(case["solver"], bits=case["bits"]), bodies=bodies)
    if kind == "frames":
        if case["scene"] == "towers":
            bodies = scenes.reference_towers()
            bodies["position"][2:, 0] += rng.uniform(-0.01, 0.01, len(bodies) - 2).astype(np.float32)
        else:
            s = case["side"]
            bodies = scenes.cubes_grid(seed, s, s, s)
        world = beatbox.RigidBodyManager(_desc(case["solver"], case["iterations"], 30, AWAKE))
        world.build_accel_structs(bodies)
        world.simulate(150)  # the drop onto the ground is behind it
        return dict(case=case, world=world)
    if kind == "serve":
        sizes = _spread(case["requests"], case["lo"], case["hi"], rng)
        steps = rng.permutation(np.rint(np.linspace(case["steps_lo"], case["steps_hi"], len(sizes))).astype(int))
        requests = [(scenes.serving_pile(seed * 1000 + k, int(n)), int(s)) for k, (n, s) in enumerate(zip(sizes, steps))]
        server = beatbox.Server(budget_bytes=24 << 30, max_worlds=256, max_resident_bodies=200_000, team_bodies=4096,
                                split_bodies=256)
        return dict(case=case, server=server, requests=requests, desc=_desc("avbd", 10))
    batch = beatbox.Batch()
    if kind == "pile":
        worlds = [(_desc("avbd", 10), _pile(seed, case["bodies"]))]
    elif kind == "gas":
        d = _desc("pgs_soft")
        d.gravity = 0.0
        n = case["bodies"]
        worlds = [(d, scenes.sphere_gas(seed, n, half=500.0 * (n / 1e6) ** (1 / 3)))]
    elif kind == "batch":
        d = _desc(case["solver"])
        sizes = _spread(case["worlds"], case["lo"], case["hi"], rng)
        halves = rng.uniform(0.3, 0.7, len(sizes))
        worlds = [(d, _stack_world(int(n), float(h), w % 2 == 0)) for w, (n, h) in enumerate(zip(sizes, halves))]
        batch.set_param(beatbox.PARAM_PAIR_SCALE, 2)
    else:
        d = _desc("avbd", 10)
        batch.set_param(beatbox.PARAM_PAIR_SCALE, 2)
        for cells in scenes.VOXEL_SHAPES.values():
            batch.add_voxel_shape(cells, scenes.VOXEL_SIZE, scenes.VOXEL_DENSITY)
        worlds = [(d, scenes.voxel_mixed_pile(seed * 100 + k, case["bodies"])[1]) for k in range(case["worlds"])]
    for d, bodies in worlds:
        batch.add_world(d, bodies)
    tune = kind in ("pile", "gas") or (kind == "batch" and case["solver"] == "pgs_soft")
    return dict(case=case, step=_Stepped(batch, [len(b) for _, b in worlds], 10, tune))


def _pile(seed, n):
    # the 100,000-body column's density at any size
    s = (n / 100_000) ** (1 / 3)
    return scenes._mixed_pile(seed, n, 0.25, 1.0, 30.0 * s, 1.0, 1.0 + 200.0 * s)


def _fields(b):
    return {k: b[k].astype(np.int64) if b[k].dtype.kind == "u" else b[k] for k in b.dtype.names}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "fresh":
        code, bodies, _ = beatbox.step_noalloc(state["desc"], state["bodies"], case["steps"])
        return {"code": code, **_fields(bodies)}
    if kind == "frames":
        world = state["world"]
        for _ in range(case["frames"]):
            world.simulate(1)
            stats = world.read_back_sim_config()
            bodies = world.read_bodies()
        return {"stats": np.array(list(stats.values()), np.int64), **_fields(bodies)}
    if kind == "serve":
        server = state["server"]
        tickets = [(server.submit(state["desc"], b, steps), len(b)) for b, steps in state["requests"]]
        server.drain()
        done = [server.poll(t, n) for t, n in tickets]
        return {"state": np.array([s for s, _, _ in done], np.int64), **_fields(np.concatenate([b for _, b, _ in done]))}
    step = state["step"]
    step.batch.step(case["steps"], use_graph=True)
    for w, n, p in step.targets:
        step.batch.instance_transforms(w, n, p)
    return step.poses


# Contacts and manifolds per body of each kind's scenes, as stepping them
# shows them; the sizes of work() follow from these.
_PER_BODY = {"fresh": (1.5, 0.6), "frames": (5.0, 1.5), "pile": (4.0, 2.5), "gas": (0.01, 0.01), "batch": (4.5, 1.2),
             "voxel": (4.0, 1.5), "serve": (3.0, 2.0)}


def work(case):
    """Per body and step the row read and written once (88 bytes each way)
    and the properties read (96); per contact the warm-start state read and
    written (100 bytes each way), per manifold its header (64).  Operations:
    about 300 per contact and sweep of the PGS family (2 I + 1 sweeps), 900
    per contact and sweep of AVBD (14 primal, 10 dual at half), 600 per
    manifold for the contact test."""
    kind, solver = case["kind"], case.get("solver", "avbd")
    if kind == "serve":
        n = sum(_spread(case["requests"], case["lo"], case["hi"], np.random.default_rng(0)))
        steps = (case["steps_lo"] + case["steps_hi"]) / 2
    elif kind == "batch":
        n = int(sum(_spread(case["worlds"], case["lo"], case["hi"], np.random.default_rng(0)))) + case["worlds"]
        steps = case["steps"]
    elif kind == "frames":
        n = case["side"] ** 3 + 1 if case["scene"] == "cubes" else 27
        steps = case["frames"]
    else:
        n = case["bodies"] * case.get("worlds", 1)
        steps = case["steps"]
    if kind == "gas":
        solver = "pgs_soft"
    contacts, manifolds = (n * x for x in _PER_BODY[kind])
    sweeps = {"avbd": (14 + 5) * 900, "pgs": (case.get("iterations", 8) + 1) * 300,
              "pgs_soft": (2 * case.get("iterations", 8) + 1) * 300}[solver]
    return {"bytes": float(steps * (n * (2 * 88 + 96) + contacts * 200 + manifolds * 128) + 48 * n),
            "flops": float(steps * (contacts * sweeps + manifolds * 600 + n * 400))}


def exact(case, seed):
    """None: what a step computes is decided by its single-precision branches
    (which axis separates least, which old contact a new one continues, which
    impulse is clamped, who sleeps).  In 64 bits some of them fall the other
    way, and from there the motion is another one, so the outputs have no
    64-bit value to be compared with."""
    return None
