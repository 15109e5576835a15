"""The PGS sweeps' two forms (a row per quad of lanes, a row per lane) and the
places their body rows can lie (all in LDS, some, none) give the oracle's
bits: sizes around a wave of quads, a workgroup of quads and a second round,
the flags that change the contact's arithmetic, manifolds of more than four
contacts and the rows past the last colour, which are solved in turn."""
from __future__ import annotations

import numpy as np
import pytest

import beatbox
import scenes
from oracle_bind import OracleWorld

pytestmark = pytest.mark.gpu

FIELDS = ("position", "rotation", "velocity", "omega", "flags")
ACCUM, FRICTION = 1, 2


def _flags():
    f = scenes.SIM_DEFAULT_FLAGS
    return (f, f & ~ACCUM, f & ~FRICTION, f & ~(ACCUM | FRICTION))


@pytest.mark.parametrize("pgs_block,lds,quads", [(64, 0, 0), (64, 16, 1), (128, 512, 0), (256, 40, 1), (512, 512, 1),
                                                 (1024, 64, 0)])
def test_sweep_forms_equal_oracle(pgs_block, lds, quads):
    sizes = (1, 9, 17, 40, 70, 150, 260)
    b = beatbox.Batch()
    b.set_param(beatbox.PARAM_BLOCK, 256)
    b.set_param(beatbox.PARAM_PGS_BLOCK, pgs_block)
    b.set_param(beatbox.PARAM_PGS_LDS_ROWS, lds)
    b.set_param(beatbox.PARAM_PGS_PREFETCH, quads)
    oracles = []
    for k, n in enumerate(sizes):
        for m, flags in enumerate(_flags()):
            solver = scenes.SOLVER_PGS if (k + m) % 3 == 0 else scenes.SOLVER_PGS_SOFT
            if solver == scenes.SOLVER_PGS:  # plain PGS: the per-island path
                flags &= ~scenes.SIM_USE_GRAPH_COLORING
            d = beatbox.WorldDesc.make(**scenes.world_desc(solver=solver, iterations=3 + m, flags=flags,
                                                           morton_bits=63, quirks=0))
            bodies = scenes.random_boxes(100 + 10 * k + m, n, extent=max(1.0, 0.5 * n ** 0.5), y0=0.55, y1=2.5)
            b.add_world(d, bodies)
            o = OracleWorld(d)
            o.add_bodies(bodies)
            oracles.append((o, len(bodies)))
    # 300 more worlds make the launch a crowded one: ranges over a wave of
    # quads go to single lanes
    tiny = beatbox.WorldDesc.make(**scenes.world_desc(iterations=2, morton_bits=63, quirks=0))
    for k in range(300):
        b.add_world(tiny, scenes.random_boxes(5000 + k, 2, extent=0.6, y0=0.55, y1=1.5))
    for steps in (1, 4):
        b.step(steps)
        b.sync(allow_overflow=True)
        for w, (o, n) in enumerate(oracles):
            o.step(steps)
            g, r = b.read_world(w, n), o.read_bodies()
            for f in FIELDS:
                assert np.array_equal(g[f], r[f]), (w, n, f)


@pytest.mark.parametrize("worlds,lds", [(4, 512), (300, 0), (300, 100)])
def test_rows_past_the_colours_equal_oracle(worlds, lds):
    """Spheres closer than their radius need more colours than there are, with
    each of the flags, in a lone launch and in a crowded one."""
    b = beatbox.Batch()
    b.set_param(beatbox.PARAM_BLOCK, 256)
    b.set_param(beatbox.PARAM_PAIR_SCALE, 8)
    b.set_param(beatbox.PARAM_LANE_BODIES, 0)
    b.set_param(beatbox.PARAM_PGS_LDS_ROWS, lds)
    bodies = scenes.dense_spheres(0xBB92, side=6)
    oracles = []
    for flags in _flags():
        d = beatbox.WorldDesc.make(**scenes.world_desc(iterations=3, flags=flags, morton_bits=63, quirks=0,
                                                       gravity=0.0))
        b.add_world(d, bodies)
        o = OracleWorld(d)
        o.add_bodies(bodies)
        oracles.append(o)
    tiny = beatbox.WorldDesc.make(**scenes.world_desc(iterations=2, morton_bits=63, quirks=0))
    for k in range(worlds - len(oracles)):
        b.add_world(tiny, scenes.random_boxes(5000 + k, 2, extent=0.6, y0=0.55, y1=1.5))
    for step in range(2):
        b.step(1)
        b.sync()
        for w, o in enumerate(oracles):
            o.step(1)
            assert step or o.stats()["graph_color_overflow"] > 0
            g, r = b.read_world(w, len(bodies)), o.read_bodies()
            for f in FIELDS:
                assert np.array_equal(g[f], r[f]), (step, w, f)


@pytest.mark.parametrize("others", [False, True])
def test_one_launch_step_with_flags_equals_oracle(others):
    """BB_PARAM_FUSED with worlds of the usual flags, and of every set of
    them (which the batch then runs by stages)."""
    b = beatbox.Batch()
    b.set_param(beatbox.PARAM_FUSED, 1)
    oracles = []
    for k, flags in enumerate(_flags() if others else _flags()[:1] * 2):
        d = beatbox.WorldDesc.make(**scenes.world_desc(iterations=4, flags=flags, morton_bits=63, quirks=0))
        bodies = scenes.random_boxes(300 + k, 60 + k, extent=2.5, y0=0.55, y1=3.0)
        b.add_world(d, bodies)
        o = OracleWorld(d)
        o.add_bodies(bodies)
        oracles.append((o, len(bodies)))
    for steps in (1, 6):
        b.step(steps, use_graph=steps > 1)
        b.sync()
        for w, (o, n) in enumerate(oracles):
            o.step(steps)
            g, r = b.read_world(w, n), o.read_bodies()
            for f in FIELDS:
                assert np.array_equal(g[f], r[f]), (w, n, f)


def test_changed_flags_equal_oracle():
    """A world whose flags change between steps: the launch sequence follows
    (usual colour sweeps, those without friction or accumulation, the
    per-island path)."""
    d = beatbox.WorldDesc.make(**scenes.world_desc(iterations=4, morton_bits=63, quirks=0))
    bodies = scenes.random_boxes(77, 40, extent=2.0, y0=0.55, y1=2.5)
    w, o = beatbox.RigidBodyManager(d), OracleWorld(d)
    w.add_bodies(bodies)
    o.add_bodies(bodies)
    for flags in (scenes.SIM_DEFAULT_FLAGS, *_flags(), scenes.SIM_DEFAULT_FLAGS & ~scenes.SIM_USE_GRAPH_COLORING,
                  scenes.SIM_DEFAULT_FLAGS):
        w.clear_sim_flags(0xFFFFFFFF)
        w.set_sim_flags(flags)
        o.set_flags(flags)
        w.simulate(4)
        o.step(4)
        g, r = w.read_bodies(), o.read_bodies()
        for f in FIELDS:
            assert np.array_equal(g[f], r[f]), (flags, f)


def _plate(n: int):
    """A dynamic plate on the ground under n spheres: the plate's contacts
    take several rounds of its group."""
    bodies = scenes.random_boxes(1, 1, extent=0.1, y0=0.55, y1=0.56, half=0.5, tilt=False)
    bodies[1]["minimum"] = (-4.0, -0.25, -4.0)
    bodies[1]["maximum"] = (4.0, 0.25, 4.0)
    bodies[1]["position"] = (0.0, 0.249, 0.0)
    bodies[1]["mass"] = 8.0
    top = np.zeros(n, scenes.BODY_DESC)
    k = np.arange(n)
    top["shape"] = scenes.SHAPE_SPHERE
    top["flags"] = scenes.BODY_DYNAMIC | scenes.BODY_GRAVITY
    top["position"] = np.stack([0.5 * (k % 14) - 3.3, 0.69 + 0.0 * k, 0.5 * (k // 14) - 3.3], 1)
    top["rotation"] = (0.0, 0.0, 0.0, 1.0)
    top["radius"] = 0.2
    top["minimum"], top["maximum"] = -0.2, 0.2
    top["mass"], top["friction"] = 0.1, 0.5
    return np.concatenate([bodies, top])


@pytest.mark.parametrize("block,team,fused,more", [
    (128, 0, 0, 0), (256, 0, 1, 0), (512, 0, 0, 0), (1024, 0, 0, 0), (256, 9, 0, 0),
    (512, 0, 0, 300), (128, 0, 1, 0), (512, 0, 1, 0), (1024, 0, 1, 0)])
def test_avbd_groups_equal_oracle(block, team, fused, more):
    """Bodies solved by groups of eight lanes: one contact and several
    rounds of them per body, sizes around a workgroup's groups, both inertia
    conventions, every workgroup size (512 threads run the stage with 1,024
    up to 256 worlds, so once with 300 more), the one-launch step and workgroup
    teams."""
    b = beatbox.Batch()
    b.set_param(beatbox.PARAM_BLOCK, block)
    b.set_param(beatbox.PARAM_TEAM_BODIES, team)
    b.set_param(beatbox.PARAM_FUSED, fused)
    b.set_param(beatbox.PARAM_LANE_BODIES, 0)
    scenes_ = [_plate(1), _plate(9), _plate(170)] + [
        scenes.random_boxes(200 + n, n, extent=max(1.0, 0.4 * n ** 0.5), y0=0.55, y1=3.0) for n in (8, 33, 129)]
    oracles = []
    for k, bodies in enumerate(scenes_):
        for bits in (30, 63):
            d = beatbox.WorldDesc.make(**scenes.world_desc(solver=scenes.SOLVER_AVBD, iterations=10, morton_bits=bits,
                                                           quirks=scenes.QUIRKS_PARITY if bits == 30 else 0))
            b.add_world(d, bodies)
            o = OracleWorld(d)
            o.add_bodies(bodies)
            oracles.append((o, len(bodies)))
    tiny = beatbox.WorldDesc.make(**scenes.world_desc(solver=scenes.SOLVER_AVBD, iterations=2, morton_bits=63,
                                                      quirks=0))
    for k in range(more):
        b.add_world(tiny, scenes.random_boxes(5000 + k, 2, extent=0.6, y0=0.55, y1=1.5))
    for steps in (1, 5):
        b.step(steps)
        b.sync(allow_overflow=True)
        for w, (o, n) in enumerate(oracles):
            o.step(steps)
            g, r = b.read_world(w, n), o.read_bodies()
            for f in FIELDS:
                assert np.array_equal(g[f], r[f]), (w, n, f)


@pytest.mark.parametrize("team", [0, 9])
def test_avbd_sleeping_worlds_equal_oracle(team):
    """Worlds that fall asleep, wholly or but for a box that drops among the
    sleepers: manifolds between rows that do not move take no part in the
    sweeps."""
    b = beatbox.Batch()
    b.set_param(beatbox.PARAM_BLOCK, 256)
    b.set_param(beatbox.PARAM_TEAM_BODIES, team)
    b.set_param(beatbox.PARAM_LANE_BODIES, 0)
    d = beatbox.WorldDesc.make(**scenes.world_desc(solver=scenes.SOLVER_AVBD, iterations=10, morton_bits=63, quirks=0))
    oracles, asleep = [], [0, 0]
    for late in (False, True):
        bodies = scenes.random_boxes(61, 12, extent=1.5, y0=0.55, y1=2.0)
        if late:
            bodies[-1]["position"] = (0.1, 16.0, 0.2)
        b.add_world(d, bodies)
        o = OracleWorld(d)
        o.add_bodies(bodies)
        oracles.append((o, len(bodies)))
    for _ in range(24):
        b.step(10)
        b.sync()
        for w, (o, n) in enumerate(oracles):
            o.step(10)
            g, r = b.read_world(w, n), o.read_bodies()
            for f in FIELDS:
                assert np.array_equal(g[f], r[f]), (w, f)
            asleep[w] = max(asleep[w], o.stats()["sleeping_count"])
    assert min(asleep) > 0, asleep


@pytest.mark.parametrize("team", [0, 9])
def test_avbd_lists_without_partners_equal_oracle(team):
    """Plates pressed into each other, eight contacts a pair: the body lists
    have more entries than there is room for the other rows beside them."""
    m = 20
    rng = np.random.default_rng(3)
    bodies = np.zeros(m, scenes.BODY_DESC)
    bodies["shape"] = scenes.SHAPE_BOX
    bodies["flags"] = scenes.BODY_DYNAMIC
    bodies["position"][:, 1] = 0.004 * np.arange(m)
    bodies["rotation"] = scenes.yaw_quat(rng.uniform(0.0, np.pi / 2, m))
    bodies["minimum"], bodies["maximum"] = (-1.0, -0.1, -1.0), (1.0, 0.1, 1.0)
    bodies["mass"], bodies["friction"] = 1.0, 0.5
    d = beatbox.WorldDesc.make(**scenes.world_desc(solver=scenes.SOLVER_AVBD, iterations=10, morton_bits=63, quirks=0,
                                                   gravity=0.0))
    b, o = beatbox.Batch(), OracleWorld(d)
    b.set_param(beatbox.PARAM_TEAM_BODIES, team)
    b.add_world(d, bodies)
    o.add_bodies(bodies)
    for step in range(3):
        b.step(1)
        b.sync()
        o.step(1)
        # two entries a contact, eight a pair slot (8 m + 64) beside the partners
        assert step or 2 * o.stats()["contact_count"] > 8 * (8 * m + 64)
        g, r = b.read_world(0, m), o.read_bodies()
        for f in FIELDS:
            assert np.array_equal(g[f], r[f]), (step, f)
