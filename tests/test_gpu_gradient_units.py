"""Pressure gradient and wall term on both sides of the sizes where the 3D
kernel changes its work units and lanes per particle, with units cut off at the
domain's end, and with particles far outside their (border) cells, whose units
take the global-memory path (needs an MI355X).  Against FP64 sums over k-d
trees' neighbours for a sample of particles, within 4e-6 (FP32 terms of a few
roundings each, with distances accurate to 1e-7 H) of the sum of the terms'
magnitudes with the kernel's largest slope, and FP32's rounding of v."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

from vps import Projection, scenes, _abi

pytestmark = pytest.mark.gpu

DX = 1.0 / 64


def spline(r, h):
    x = r / h
    c0 = 8 / (np.pi * h ** 3)
    w = c0 * np.where(x < .5, 6 * x * x * (x - 1) + 1, 2 * np.maximum(1 - x, 0) ** 3)
    dw = 6 * c0 / h * np.where(x < .5, x * (3 * x - 2), -np.maximum(1 - x, 0) ** 2)
    return w, dw


# 2 x 2 x 2 cells up to 32,000 particles, 4 x 2 x 2 up to 250,000
@pytest.mark.parametrize("block,cut", [
    ((5, 4, 3), None), ((31, 32, 32), None), ((32, 32, 32), None),
    ((62, 63, 64), None), ((63, 63, 63), None), ((12, 11, 13), 0.6), ((33, 32, 32), 0.6),
    ((63, 64, 65), 0.7)])
def test_velocity_update(block, cut):
    sc = scenes.dam_break(3, DX, [(b + 4) * DX for b in block], [b * DX for b in block])
    rng = np.random.default_rng(4)
    if cut:   # the last cells of the x axis also hold everything beyond them
        sc["domain_hi"] = sc["domain_hi"].copy()
        sc["domain_hi"][0] = cut * block[0] * DX
    v = rng.normal(size=sc["x"].shape).astype(np.float32).astype(np.float64)
    bv = rng.normal(size=sc["bx"].shape).astype(np.float32).astype(np.float64)
    sc = dict(sc, v=v, bv=bv)
    g = Projection(sc, rest_density_mode=_abi.FROM_PARAMS, kappa_mode=_abi.FROM_PARAMS)
    g.initialize()
    bvol = g.boundary_fields()[1]
    g.project()
    x, after = g.particles()
    virt = g.virtual()
    dims, lin = sc["lattice_dims"], virt["node"]
    nodes = np.asarray(sc["lattice_origin"])[:3] + sc["lattice_spacing"] * np.stack(
        [lin % dims[0], lin // dims[0] % dims[1], lin // dims[0] // dims[1]], axis=1)
    q = virt["vol"] * virt["p"]
    h, H = 4 * sc["particle_radius"], 4 * sc["lattice_spacing"]
    slope = 2 * 8 / (np.pi * H ** 4)                     # |W'| at its largest
    tn, tb = cKDTree(nodes), cKDTree(sc["bx"])
    pick = rng.choice(len(x), min(len(x), 600), replace=False)
    for i in pick:
        J = np.asarray(tn.query_ball_point(x[i], H), dtype=int)
        d = x[i] - nodes[J]
        r = np.linalg.norm(d, axis=1)
        f = (d * (-q[J] * spline(r, H)[1] / np.where(r > 0, r, 1))[:, None]).sum(0)
        b = np.asarray(tb.query_ball_point(x[i], h), dtype=int)
        rel = v[i] - bv[b]
        dn = np.minimum((sc["bn"][b] * rel).sum(1), 0)
        w = bvol[b] * spline(np.linalg.norm(x[i] - sc["bx"][b], axis=1), h)[0]
        f -= ((w * dn)[:, None] * sc["bn"][b]).sum(0)
        tol = 4e-6 * (np.abs(q[J]).sum() * slope + (w * np.linalg.norm(rel, axis=1)).sum())
        assert np.all(np.abs(after[i] - v[i] - f) <= tol + 2.0 ** -23 * np.abs(v[i]))
    g.close()
