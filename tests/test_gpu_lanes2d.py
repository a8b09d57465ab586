"""The 2D walks (density, viscosity, virtual sums, gradient) on both sides of
the size where they give up four lanes per particle or node, and at a few small
and odd ones (needs an MI355X).  Density, virtual set, rho and V against the FP64
oracle with the bars of the parity tests; viscosity and gradient against FP64
sums over k-d trees' neighbours, within 4e-6 (FP32 terms of a few roundings each)
of the sum of the terms' magnitudes and FP32's rounding of the velocity."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

import oracle_py as O
from vps import Projection, scenes, _abi

pytestmark = pytest.mark.gpu

DX = 1.0 / 256
MODES = dict(rest_density_mode=_abi.FROM_PARAMS, kappa_mode=_abi.FROM_PARAMS)


def spline(r, h):
    x = r / h
    c0 = 40 / (7 * np.pi * h ** 2)
    w = c0 * np.where(x < .5, 6 * x * x * (x - 1) + 1, 2 * np.maximum(1 - x, 0) ** 3)
    dw = 6 * c0 / h * np.where(x < .5, x * (3 * x - 2), -np.maximum(1 - x, 0) ** 2)
    return w, dw


# four lanes up to 130,000 particles
@pytest.mark.parametrize("block", [(5, 4), (17, 31), (101, 67), (360, 361), (361, 361)])
def test_2d_walks(block):
    sc = scenes.dam_break(2, DX, [(b + 6) * DX for b in block], [b * DX for b in block])
    rng = np.random.default_rng(6)
    sc["v"] = rng.normal(size=sc["x"].shape).astype(np.float32).astype(np.float64)
    sc["bv"] = rng.normal(size=sc["bx"].shape).astype(np.float32).astype(np.float64)
    o = O.Oracle(sc, **MODES)
    o.initialize()
    g = Projection(sc, **MODES)
    g.initialize()
    rho = g.real_fields()[0]
    assert np.max(np.abs(rho / o.real_fields()[0] - 1)) < 2e-6
    vo, vg = o.virtual(), g.virtual()
    o.close()
    assert np.array_equal(vo["node"], vg["node"])
    for f in ("rho", "vol"):
        assert np.max(np.abs(vg[f] / vo[f] - 1)) < 5e-6, f

    x, v, m = sc["x"], sc["v"], sc["mass"]
    h, H = 4 * sc["particle_radius"], 4 * sc["lattice_spacing"]
    nu, dt = 0.01, 1e-4
    tree = cKDTree(x)
    pick = rng.choice(len(x), min(len(x), 500), replace=False)
    g.L.vps_apply_viscosity(g.h, dt, nu)
    v1 = g.particles()[1]
    for i in pick:
        js = np.asarray(tree.query_ball_point(x[i], h))
        js = js[js != i]
        d = x[js] - x[i]
        r = np.linalg.norm(d, axis=1)
        c = ((v[js] - v[i]) * d).sum(1) / r ** 2 * (-spline(r, h)[1] / r) / rho[js]
        terms = nu * dt * 2 * 4 * m * c[:, None] * d
        tol = 4e-6 * np.abs(terms).sum(0) + 2.0 ** -23 * np.abs(v[i])
        assert np.all(np.abs(v1[i] - (v[i] + terms.sum(0))) <= tol)

    bvol = g.boundary_fields()[1]
    g.project()
    v2 = g.particles()[1]
    virt = g.virtual()
    nx = sc["lattice_dims"][0]
    nodes = np.asarray(sc["lattice_origin"])[:2] + sc["lattice_spacing"] * np.stack(
        [virt["node"] % nx, virt["node"] // nx], axis=1)
    q = virt["vol"] * virt["p"]
    slope = 2 * 40 / (7 * np.pi * H ** 3)
    tn, tb = cKDTree(nodes), cKDTree(sc["bx"])
    for i in pick:
        J = np.asarray(tn.query_ball_point(x[i], H), dtype=int)
        d = x[i] - nodes[J]
        r = np.linalg.norm(d, axis=1)
        f = (d * (-q[J] * spline(r, H)[1] / np.where(r > 0, r, 1))[:, None]).sum(0)
        b = np.asarray(tb.query_ball_point(x[i], h), dtype=int)
        rel = v1[i] - sc["bv"][b]
        w = bvol[b] * spline(np.linalg.norm(x[i] - sc["bx"][b], axis=1), h)[0]
        f -= ((w * np.minimum((sc["bn"][b] * rel).sum(1), 0))[:, None] * sc["bn"][b]).sum(0)
        tol = 4e-6 * (np.abs(q[J]).sum() * slope + (w * np.linalg.norm(rel, axis=1)).sum())
        assert np.all(np.abs(v2[i] - v1[i] - f) <= tol + 2.0 ** -23 * np.abs(v1[i]))
    g.close()
