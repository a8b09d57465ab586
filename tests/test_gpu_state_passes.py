"""Particle sets beyond the bounded staging of the host state (needs an MI355X):
512 MB, so 11,184,810 particles in 3D go in one pass and more in several.  Upload
of a new set, read-back in caller order from the cell-sorted state, overwriting
a resident set, refusals that leave the state alone, and the device memory that
the context keeps: 140 bytes a particle of state and sort scratch, the staging,
and tables that stay below 128 MB here."""
import ctypes as C

import numpy as np
import pytest

from vps import Projection, VpsError, _abi, scenes

pytestmark = pytest.mark.gpu

PASS = (512 << 20) // 48


def free_memory():
    hip = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def scene(n):
    """n random particles, eight to a cell, a few walls, a lattice of one brick."""
    rng = np.random.default_rng(31)
    x = rng.random((n, 3))
    v = rng.random((n, 3), dtype=np.float32).astype(np.float64)
    wall = np.full((4, 3), 0.5)
    sc = scenes.grain_scene(x, v, (8 / n) ** (1 / 3) / 4, wall, np.ones_like(wall),
                            np.zeros_like(wall), np.zeros(3), np.ones(3))
    return dict(sc, lattice_dims=np.full(3, 8))


@pytest.mark.parametrize("n", [PASS, PASS + 1, 20_000_000])
def test_set_and_get(n):
    sc = scene(n)
    Projection(scenes.small_3d(12, 8, 6)).close()   # (the runtime's own memory)
    before = free_memory()
    g = Projection(sc)
    held = before - free_memory()
    assert held < 140 * n + (512 << 20) + (128 << 20)
    x, v = g.particles()
    assert np.array_equal(x, sc["x"]) and np.array_equal(v, sc["v"])
    g.initialize()   # sorted by cell from here on
    x, v = g.particles()
    assert np.array_equal(x, sc["x"]) and np.array_equal(v, sc["v"])
    vol = g.real_fields()[1]
    x2, v2 = sc["x"][::-1].copy(), -sc["v"]
    for i in (0, n - 1):
        bad = x2.copy()
        bad[i, 1] = np.nan
        with pytest.raises(VpsError) as e:
            g.set_particles(bad, v2)
        assert e.value.code == _abi.VPS_ERR_NONFINITE
    del bad
    x, v = g.particles()
    assert np.array_equal(x, sc["x"]) and np.array_equal(v, sc["v"])
    g.set_particles(x2, v2)
    x, v = g.particles()
    assert np.array_equal(x, x2) and np.array_equal(v, v2)
    assert np.array_equal(g.real_fields()[1], vol)
    g.set_particles(sc["x"])   # velocities kept without v
    x, v = g.particles()
    assert np.array_equal(x, sc["x"]) and np.array_equal(v, v2)
    g.close()
