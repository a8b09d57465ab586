"""Few particles in a lattice of 2^20 bricks and more (needs an MI355X): the
first generation's grid covers every brick with several lanes per node, and has
to stay within the threads of a launch.  Same fields and velocities as in the
block's own lattice, whose nodes these are; bars as in the parity tests (the
sums may run in another order)."""
import numpy as np
import pytest

from vps import Projection, scenes

pytestmark = pytest.mark.gpu


def run(sc):
    g = Projection(sc)
    g.initialize()
    for _ in range(2):
        g.advect(1e-3, 9.8)
        s = g.projection_step()
    out = g.virtual(), g.particles(), s["cg_true_rel_residual"]
    g.close()
    return out


@pytest.mark.parametrize("nz", [512, 513])   # 2^20 bricks, and 2^20 + 2^14
def test_few_particles_in_a_large_lattice(nz):
    sc = scenes.small_3d(12, 8, 6)
    v0, (x0, u0), _ = run(sc)
    dims = np.array([1024, 1024, nz])
    large = dict(sc, lattice_dims=dims)
    large["domain_hi"] = sc["domain_lo"] + (dims + 8) * sc["lattice_spacing"]
    v1, (x1, u1), res = run(large)

    def coords(lin, d):
        return np.stack([lin % d[0], lin // d[0] % d[1], lin // d[0] // d[1]])
    assert np.array_equal(coords(v0["node"], sc["lattice_dims"]), coords(v1["node"], dims))
    assert np.max(np.abs(v1["rho"] / v0["rho"] - 1)) < 5e-6
    assert res < 1e-6
    assert np.max(np.abs(x1 - x0)) < 1e-6
    assert np.linalg.norm(u1 - u0) < 1e-4 * np.linalg.norm(u0)
