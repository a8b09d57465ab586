"""Contexts of their own on several host threads (needs an MI355X): created, run
and destroyed at the same time, each gives what it gives alone, bit for bit."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from vps import Projection, scenes

pytestmark = pytest.mark.gpu


def run(sc):
    g = Projection(sc)
    g.initialize()
    for _ in range(6):
        g.advance(5e-4, 9.8, 0.01, scenes.box_colliders(sc), True)
    out = g.particles()
    g.close()
    return out


def test_contexts_on_threads():
    scs = [scenes.small_2d(20), scenes.small_3d(12, 8, 6), scenes.small_2d(37),
           scenes.small_3d(16, 16, 12)] * 2
    alone = [run(sc) for sc in scs[:4]]
    with ThreadPoolExecutor(len(scs)) as pool:
        together = list(pool.map(run, scs))
    for i, (x, v) in enumerate(together):
        assert np.array_equal(x, alone[i % 4][0]) and np.array_equal(v, alone[i % 4][1])
