"""The grains' contact walk where it changes (needs an MI355X), against the
FP64 oracle with the bars of the DEM parity test: few grains (blocks and
waves partly filled, every grain or none next to a wall), rows of cells with
more than 32 candidates (the row-by-row walk), grains on cell faces, and
grains outside the domain (clamped into border cells)."""
import numpy as np
import pytest

import oracle_py as O
from vps import DemSand, scenes

pytestmark = pytest.mark.gpu

YOUNG, POISSON, PHI = 1e5, 0.3, 0.5
R = 0.0125


def build(kind, dim):
    rng = np.random.default_rng(17)
    box = np.full(dim, 40 * 2 * R)
    w, wn, wv = scenes._box_walls(dim, 2 * R, box, 3)
    lo, hi = np.zeros(3), np.zeros(3)
    lo[:dim], hi[:dim] = -12 * R, box + 12 * R
    if kind.startswith("few"):
        n = int(kind[3:])
        x = rng.uniform(4 * R, 10 * R if n < 5 else 30 * R, size=(n, dim))
    elif kind == "bulk":       # no grain next to a wall
        x = rng.uniform(20 * R, 36 * R, size=(700, dim))
    elif kind == "dense":      # about 75 grains a cell
        x = rng.uniform(2 * R, 14 * R, size=(2000 if dim == 3 else 700, dim))
    elif kind == "faces":      # on the faces of the cells, and half a cell off
        m = 9
        g = np.meshgrid(*[np.arange(m) * 2 * R for _ in range(dim)], indexing="ij")
        x = np.stack([a.reshape(-1) for a in g], 1) + lo[:dim] + 16 * R
    else:                      # outside: a domain smaller than the set
        x = rng.uniform(0, 24 * R, size=(900, dim))
        lo[:dim], hi[:dim] = 4 * R, 16 * R
    v = 0.2 * rng.normal(size=x.shape)
    return scenes.grain_scene(x, v, R, w, wn, wv, lo, hi)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("kind", ["few1", "few2", "few65", "few300", "bulk", "dense", "faces",
                                  "outside"])
def test_contact_walk(kind, dim):
    gs = build(kind, dim)
    g = DemSand(gs, young=YOUNG, poisson=POISSON, friction_angle=PHI)
    o = O.Oracle(gs)
    dt = 1e-4
    for step in range(2):
        x0, v0 = g.particles()
        o.set_particles(x0, v0)
        g.advance(dt)
        o.dem_step(dt, 9.8, YOUNG, POISSON, PHI)
        xg, vg = g.particles()
        xo, vo = o.particles()
        assert np.array_equal(xg, xo), step
        dv = np.abs(vo - v0).max()
        assert np.linalg.norm(vg - vo) / np.linalg.norm(vo) < 1e-4, step
        assert np.abs(vg - vo).max() / dv < 1e-4, step
    g.close()
    o.close()
