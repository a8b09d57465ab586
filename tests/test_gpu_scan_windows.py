"""The one-launch scan at its larger tiles and beyond one look-back window (needs
an MI355X).  Tiles hold 2,048 elements up to 524,288, 4,096 up to 4,194,304 and
8,192 above; a look-back reads the 1,024 tiles before one at a time, so it can
need a second window from 8,388,609 elements on, and the column scan (256 a tile)
from 262,145 columns."""
import numpy as np
import pytest

import sampling_oracle as S
from vps import Projection, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [524289, 4096 * 129 - 1, 4096 * 129, 4096 * 129 + 1, 4194304,
                               4194305, 8192 * 513, 8192 * 1024, 8192 * 1025 + 5])
def test_scan_sizes(n):
    """One row of candidates, of which a sphere keeps a stretch, compacted by the
    scan: bit for bit the sampling oracle's."""
    r = 0.01
    e = np.zeros((0, 2))
    lo, hi = np.array([-1.0 - n * r, -0.4, 0]), np.array([1.0 + n * r, 0.1, 0])
    g = Projection(scenes.grain_scene(np.zeros((1, 2)), np.zeros((1, 2)), r, e, e, e, lo, hi))
    center, half = np.array([0.1, -0.2]), np.array([n * r, r])
    s = (S.SPHERE, [0.1 + 0.2 * n * r, -0.2, 0], [n * r * 0.63, 0, 0], False)
    xo, no = S.add_surface(2, r, S.Surface(*s, 2), center, half)
    g.add_surface(s[0], s[1], s[2], center, half)
    x, nrm, _ = g.boundary()
    assert len(xo) > 0 and np.array_equal(x, xo) and np.array_equal(nrm, no)
    g.close()


@pytest.mark.parametrize("side", [4096, 4104])   # 512 x 512 columns, and 513 x 513
def test_column_scan(side):
    """A block in the last columns of a wide lattice: the fields and velocities of
    its own lattice, whose nodes these are but for the rounding of their
    coordinates; bars as in the parity tests."""
    sc = scenes.small_3d(12, 8, 6)
    wide = dict(sc, lattice_dims=np.array([side, side, sc["lattice_dims"][2]]))
    shift = (wide["lattice_dims"] - sc["lattice_dims"]) * sc["lattice_spacing"]
    wide["lattice_origin"] = sc["lattice_origin"] - shift
    wide["domain_lo"] = sc["domain_lo"] - shift
    out = []
    for s in (sc, wide):
        g = Projection(s)
        g.initialize()
        for _ in range(2):
            g.advect(1e-3, 9.8)
            st = g.projection_step()
        out.append((g.virtual(), g.particles()[1], st))
        g.close()
    (v0, u0, s0), (v1, u1, s1) = out
    assert len(v0["node"]) == len(v1["node"])
    assert np.max(np.abs(v1["rho"] / v0["rho"] - 1)) < 5e-6
    assert abs(s1["cg_iterations"] - s0["cg_iterations"]) <= 1
    assert s1["cg_true_rel_residual"] < 1e-6
    assert np.linalg.norm(u1 - u0) < 1e-4 * np.linalg.norm(u0)
