"""The broad phase over every pair of rows (small worlds) and by several
workgroups in three launches, and the narrow phase by several workgroups per
world, give the oracle's bits: sizes around a wave, around the lines where
the tree takes over (N^2 = 40,960 per wave in three launches, 16,384 in one,
10 million over a launch of more worlds than CUs) and around the smallest world of
the three launches, voxel worlds with their expanded slots, and a row of more
partners than the tree form stages."""
from __future__ import annotations

import numpy as np
import pytest

import beatbox
import scenes
from oracle_bind import OracleWorld

pytestmark = pytest.mark.gpu

FIELDS = ("position", "rotation", "velocity", "omega", "flags")
PGS = scenes.world_desc(iterations=3, morton_bits=63, quirks=0)


def _check(b, oracles, steps=(1, 3)):
    for k in steps:
        b.step(k)
        b.sync()
        for w, (o, n) in enumerate(oracles):
            o.step(k)
            g, r = b.read_world(w, n), o.read_bodies()
            assert b.stats(w)["broad_phase_collision_count"] == o.stats()["broad_phase_collision_count"], (w, n)
            for f in FIELDS:
                assert np.array_equal(g[f], r[f]), (w, n, f)


def _worlds(b, sizes, seed):
    out = []
    for n in sizes:
        d = beatbox.WorldDesc.make(**PGS)
        bodies = scenes.random_boxes(seed + n, n - 1, extent=max(1.0, 0.45 * n ** 0.5), y0=0.55, y1=3.0)
        assert len(bodies) == n
        b.add_world(d, bodies)
        o = OracleWorld(d)
        o.add_bodies(bodies)
        out.append((o, n))
    return out


# one world takes 16 workgroups (64 waves of 256 threads: 1,619 rows), 20
# worlds take 12, 100 worlds two and the one-launch broad phase
@pytest.mark.parametrize("block,worlds,sizes", [
    (256, 1, (2,)), (256, 1, (65,)), (256, 1, (256,)), (256, 1, (257,)), (256, 1, (1619,)), (256, 1, (1620,)),
    (512, 1, (1025,)), (1024, 1, (700,)), (128, 20, (63, 64, 300)),
    (256, 100, (128, 404, 405)), (512, 100, (572, 573)), (256, 300, (180, 181, 182, 404, 600)),
    (256, 200, (256, 257)), (256, 300, (182, 183)), (128, 1024, (98, 99))])
def test_broad_and_narrow_spread_equal_oracle(block, worlds, sizes):
    b = beatbox.Batch()
    b.set_param(beatbox.PARAM_BLOCK, block)
    b.set_param(beatbox.PARAM_LANE_BODIES, 0)
    b.set_param(beatbox.PARAM_TEAM_BODIES, 0)
    b.set_param(beatbox.PARAM_FUSED, 0)
    oracles = _worlds(b, sizes, 9000)
    tiny = beatbox.WorldDesc.make(**PGS)
    for k in range(worlds - len(sizes)):
        b.add_world(tiny, scenes.random_boxes(7000 + k, 2, extent=0.6, y0=0.55, y1=1.5))
    _check(b, oracles)


@pytest.mark.parametrize("n,worlds", [(40, 1), (300, 1), (300, 300)])
def test_voxel_slots_equal_oracle(n, worlds):
    shapes, bodies = scenes.voxel_mixed_pile(0xBB90, n)
    d = beatbox.WorldDesc.make(**PGS)
    b = beatbox.Batch()
    b.set_param(beatbox.PARAM_TEAM_BODIES, 0)
    o = OracleWorld(d)
    for _, cells in shapes:
        b.add_voxel_shape(cells, scenes.VOXEL_SIZE, scenes.VOXEL_DENSITY)
        o.add_voxel_shape(cells, scenes.VOXEL_SIZE, scenes.VOXEL_DENSITY)
    b.add_world(d, bodies)
    o.add_bodies(bodies)
    for k in range(worlds - 1):
        b.add_world(d, scenes.random_boxes(7000 + k, 2, extent=0.6, y0=0.55, y1=1.5))
    _check(b, [(o, len(bodies))], steps=(1, 12))


@pytest.mark.parametrize("side", [6, 12])
def test_many_partners_equal_oracle(side):
    """Spheres closer than their radius: dozens of pairs per row (216 spheres
    compared row by row, 1,728 through the three launches' tree)."""
    bodies = scenes.dense_spheres(0xBB91, side=side)
    d = beatbox.WorldDesc.make(**scenes.world_desc(iterations=2, morton_bits=63, quirks=0, gravity=0.0))
    b = beatbox.Batch()
    b.set_param(beatbox.PARAM_BLOCK, 256)
    b.set_param(beatbox.PARAM_PAIR_SCALE, 8)
    b.set_param(beatbox.PARAM_TEAM_BODIES, 0)
    b.set_param(beatbox.PARAM_LANE_BODIES, 0)
    b.add_world(d, bodies)
    o = OracleWorld(d)
    o.add_bodies(bodies)
    _check(b, [(o, len(bodies))], steps=(1,))
