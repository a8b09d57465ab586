"""Particles in and out of a context (needs an MI355X): sizes below, at and
across the pieces of the pinned transfer, either output alone, the resident
(initialized) and the new-set upload, and non-finite input, which must leave
the state as it was.  Positions return bit for bit, velocities as FP32."""
import ctypes as C

import numpy as np
import pytest

from vps import Projection, VpsError, scenes, _abi

pytestmark = pytest.mark.gpu

PIECE = 512 << 10   # bytes


def grains(dim, n, seed=3):
    rng = np.random.default_rng(seed)
    x = rng.uniform(0.05, 0.95, size=(n, dim))
    e = np.zeros((0, dim))
    sc = scenes.grain_scene(x, rng.normal(size=(n, dim)), 0.01, e, e, e, np.zeros(3),
                            np.ones(3))
    return sc


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [1, 63, 257, 5000, PIECE // 48, PIECE // 24, PIECE // 24 + 1, 300001])
def test_round_trip(dim, n):
    sc = grains(dim, n)
    g = Projection(sc)
    x, v = g.particles()
    assert np.array_equal(x, sc["x"])
    assert np.array_equal(v, sc["v"].astype(np.float32).astype(np.float64))
    d = C.POINTER(C.c_double)
    only = np.zeros_like(x)
    assert g.L.vps_get_particles(g.h, only.ctypes.data_as(d), None) == 0
    assert np.array_equal(only, x)
    assert g.L.vps_get_particles(g.h, None, only.ctypes.data_as(d)) == 0
    assert np.array_equal(only, v)
    bad = sc["x"].copy()
    bad[n // 2, dim - 1] = np.nan
    with pytest.raises(VpsError) as e:
        g.set_particles(bad, sc["v"])
    assert e.value.code == _abi.VPS_ERR_NONFINITE
    assert np.array_equal(g.particles()[0], x)
    g.close()


@pytest.mark.parametrize("dim", [2, 3])
def test_resident_upload(dim):
    sc = scenes.small_2d(20) if dim == 2 else scenes.small_3d(12, 8, 6)
    g = Projection(sc)
    g.initialize()
    g.advance(1e-3, 9.8)
    rng = np.random.default_rng(5)
    x = sc["x"] + rng.uniform(-1e-3, 1e-3, size=sc["x"].shape)
    v = rng.normal(size=x.shape)
    vol = g.real_fields()[1]
    g.set_particles(x, v)
    for bad in (np.inf, -np.inf, np.nan):
        w = v.copy()
        w[-1, 0] = bad
        with pytest.raises(VpsError) as e:
            g.set_particles(x + 1, w)
        assert e.value.code == _abi.VPS_ERR_NONFINITE
    xg, vg = g.particles()
    assert np.array_equal(xg, x)
    assert np.array_equal(vg, v.astype(np.float32).astype(np.float64))
    assert np.array_equal(g.real_fields()[1], vol)   # frozen volumes kept
    g.set_particles(x)                               # velocities kept without v
    assert np.array_equal(g.particles()[1], vg)
    g.close()
