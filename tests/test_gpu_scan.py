"""The one-launch scan at the edges of its tiles (needs an MI355X), through
vps_add_surface: one row of candidates, of which a sphere keeps a stretch,
compacted by the scan; bit for bit against the sampling oracle.  Tiles hold
2,048 elements (8,192 above 524,288); a look-back reads 64 tiles at a time."""
import numpy as np
import pytest

import sampling_oracle as S
from vps import Projection, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 255, 2047, 2048, 2049, 4097, 2048 * 64, 2048 * 65 + 1,
                               2048 * 200 + 7, 524288, 524289, 8192 * 65, 8192 * 131 + 5])
def test_scan_sizes(n):
    r = 0.01
    e = np.zeros((0, 2))
    lo, hi = np.array([-1.0 - n * r, -0.4, 0]), np.array([1.0 + n * r, 0.1, 0])
    g = Projection(scenes.grain_scene(np.zeros((1, 2)), np.zeros((1, 2)), r, e, e, e, lo, hi))
    center, half = np.array([0.1, -0.2]), np.array([n * r, r])
    for radius in (n * r * 0.63, 2.5 * n * r):   # a part of the row, all of it
        s = (S.SPHERE, [0.1 + 0.2 * n * r, -0.2, 0], [radius, 0, 0], False)
        xo, no = S.add_surface(2, r, S.Surface(*s, 2), center, half)
        before = len(g.boundary()[0])
        g.add_surface(s[0], s[1], s[2], center, half)
        x, nrm, _ = g.boundary()
        assert len(xo) > 0 and np.array_equal(x[before:], xo)
        assert np.array_equal(nrm[before:], no)
    g.close()
