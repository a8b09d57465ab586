"""The sets that the walks sum over at every number of lanes per particle (needs
an MI355X): the counts run the kernels that a run of the size launches, and lie
between the exact sets of radius (1 -+ 1e-5) h or H, for a sample of particles."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

from vps import Projection, scenes

pytestmark = pytest.mark.gpu

DX = 1.0 / 64
BAND = 1e-5


# density and viscosity: 8 lanes up to 32,000 particles, 4 up to 400,000, 2 up to
# 900,000, then 1; gradient: 8 up to 32,000, 4 up to 250,000, then 1
@pytest.mark.parametrize("block", [(31, 32, 32), (32, 32, 32), (63, 63, 64), (74, 74, 74),
                                   (97, 97, 97)])
def test_member_counts(block):
    sc = scenes.dam_break(3, DX, [(b + 4) * DX for b in block], [b * DX for b in block])
    g = Projection(sc)
    g.initialize()
    g.projection_step()
    x = sc["x"]
    rng = np.random.default_rng(8)
    pick = np.unique(np.concatenate([rng.choice(len(x), 4000), np.arange(256),
                                     np.arange(len(x) - 256, len(x))]))
    lin, dims = g.virtual()["node"], sc["lattice_dims"]
    cell = np.stack([lin % dims[0], lin // dims[0] % dims[1], lin // dims[0] // dims[1]], axis=1)
    nodes = np.asarray(sc["lattice_origin"])[:3] + cell * sc["lattice_spacing"]
    h, H = 4 * sc["particle_radius"], 4 * sc["lattice_spacing"]
    for which, pts, radius, own in ((0, x, h, 0), (3, x, h, 1), (2, nodes, H, 0)):
        counts = g.member_counts(which)[pick] + own
        tree = cKDTree(pts)
        inner = tree.query_ball_point(x[pick], radius * (1 - BAND), return_length=True)
        outer = tree.query_ball_point(x[pick], radius * (1 + BAND), return_length=True)
        assert np.all(inner <= counts) and np.all(counts <= outer), which
    g.close()
