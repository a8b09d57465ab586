"""The pressure gradient where a unit of cells holds a particle millions of
lattice spacings away (needs an MI355X): clamped into the corner cell, its
unit's box of nodes is that large along every axis, and the product of the three
extents does not fit 64 bits (2.3e6 cubed) or 32 (2,000 cubed).  A lone
particle acts on nothing, so every other one moves as with it 60 spacings away,
bit for bit, at every unit size."""
import numpy as np
import pytest

from vps import Projection, scenes

pytestmark = pytest.mark.gpu

DX = 1.0 / 64


def velocities(block, spacings):
    sc = scenes.dam_break(3, DX, [(b + 4) * DX for b in block], [b * DX for b in block])
    sc["domain_lo"] = np.zeros(3)   # the fluid's corner lies in the corner cell
    sc["x"] = np.concatenate([sc["x"], np.full((1, 3), -spacings * DX)])
    sc["v"] = np.random.default_rng(4).normal(size=sc["x"].shape).astype(np.float32) * 1.0
    g = Projection(sc)
    g.initialize()
    s = g.projection_step()
    v = g.particles()[1]
    g.close()
    assert s["cg_true_rel_residual"] < 1e-6
    return sc["v"], v


# units of 2x2x2 cells up to 32,000 particles, 4x2x2 up to 250,000, 4x4x4 beyond
@pytest.mark.parametrize("block", [(12, 8, 6), (32, 32, 33), (63, 63, 64)])
def test_far_particle(block):
    v0, near = velocities(block, 60)
    assert not np.array_equal(near[:-1], v0[:-1])
    for spacings in (2000, 2.3e6):
        _, v = velocities(block, spacings)
        assert np.array_equal(v, near)
        assert np.array_equal(v[-1], v0[-1])
