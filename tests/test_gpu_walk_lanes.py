"""Density and viscosity on both sides of the sizes where the walks change
the number of lanes per particle (needs an MI355X), against FP64 sums over a
k-d tree's neighbours for a sample of particles.  Density within 2e-6 relative
(the bar of the parity tests); the viscous change of the velocity within 4e-6
of the sum of its terms' magnitudes (FP32 terms of a few roundings each, in
sums of about 33), plus the FP32 rounding of the velocity itself."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

from vps import Projection, scenes

pytestmark = pytest.mark.gpu


def spline(r, h):
    x = r / h
    c0 = 8 / (np.pi * h ** 3)
    w = c0 * np.where(x < .5, 6 * x * x * (x - 1) + 1, 2 * np.maximum(1 - x, 0) ** 3)
    dw = 6 * c0 / h * np.where(x < .5, x * (3 * x - 2), -np.maximum(1 - x, 0) ** 2)
    return w, dw


# 8 lanes up to 32,000 particles, 4 up to 400,000, 2 up to 900,000
@pytest.mark.parametrize("block", [(3, 3, 3), (31, 32, 32), (32, 32, 32), (73, 74, 74),
                                   (74, 74, 74), (96, 97, 96), (97, 97, 97)])
def test_density_and_viscosity(block):
    dx = 1.0 / 64
    sc = scenes.dam_break(3, dx, [(b + 4) * dx for b in block], [b * dx for b in block])
    rng = np.random.default_rng(9)
    v = rng.normal(size=sc["x"].shape).astype(np.float32).astype(np.float64)
    g = Projection(dict(sc, v=v))
    g.initialize()
    x = sc["x"]
    h, m, nu, dt = 2 * dx, sc["mass"], 0.01, 1e-4
    sample = rng.choice(len(x), min(len(x), 1500), replace=False)
    rho = g.real_fields()[0]
    tree = cKDTree(x)
    near = tree.query_ball_point(x[sample], h * (1 + 1e-9))
    need = np.unique(np.concatenate([np.asarray(k) for k in near]))
    exact = np.full(len(x), np.nan)
    for i, js in zip(need, tree.query_ball_point(x[need], h * (1 + 1e-9))):
        exact[i] = m * spline(np.linalg.norm(x[js] - x[i], axis=1), h)[0].sum()
    assert np.max(np.abs(rho[need] / exact[need] - 1)) < 2e-6
    g.L.vps_apply_viscosity(g.h, dt, nu)
    vg = g.particles()[1]
    scale = nu * dt * 2 * 5 * m
    for i, js in zip(sample, near):
        js = np.asarray(js)[np.asarray(js) != i]
        d = x[js] - x[i]
        r = np.linalg.norm(d, axis=1)
        c = ((v[js] - v[i]) * d).sum(1) / r ** 2 * (-spline(r, h)[1] / r) / exact[js]
        terms = scale * c[:, None] * d
        tol = 4e-6 * np.abs(terms).sum(0) + 2.0 ** -23 * np.abs(v[i])
        assert np.all(np.abs(vg[i] - (v[i] + terms.sum(0))) <= tol)
    g.close()
