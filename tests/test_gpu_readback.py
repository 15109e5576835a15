"""A world's readback is packed on the device and copied once: both orders,
sizes around a workgroup, the first and later worlds of a batch, before the
first step and after, and from several threads at once; steps that follow a
readback are not disturbed by it."""
from __future__ import annotations

import threading

import numpy as np
import pytest

import beatbox
import scenes
from oracle_bind import OracleWorld

pytestmark = pytest.mark.gpu

FIELDS = ("id", "position", "rotation", "velocity", "omega", "flags")


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 1000])
def test_readback_orders_equal_oracle(n):
    d = beatbox.WorldDesc.make(**scenes.world_desc(iterations=3, morton_bits=63, quirks=0))
    b = beatbox.Batch()
    oracles = []
    for k in range(3):
        bodies = scenes.random_boxes(300 + n + k, n, extent=max(1.0, 0.5 * n ** 0.5), y0=0.55, y1=2.0)[:n]
        b.add_world(d, bodies)
        o = OracleWorld(d)
        o.add_bodies(bodies)
        oracles.append(o)
    assert np.all(b.read_world(1, n)["island_index"] == 0xFFFFFFFF)
    for steps in (1, 2):
        b.step(steps)
        b.sync()
        got = [None] * 3

        def read(w):
            got[w] = (b.read_world(w, n), b.read_world(w, n, beatbox.ORDER_BY_ROW))

        threads = [threading.Thread(target=read, args=(w,)) for w in range(3)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        for w, o in enumerate(oracles):
            o.step(steps)
            ref, (by_id, by_row) = o.read_bodies(), got[w]
            for f in FIELDS:
                assert np.array_equal(by_id[f], ref[f]), (w, f)
            assert np.array_equal(by_row["row"], np.arange(n))
            assert by_row[by_id["row"]].tobytes() == by_id.tobytes(), w
