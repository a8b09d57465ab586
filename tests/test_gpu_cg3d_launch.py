"""The 3D CG iteration over the brick counts where its launch changes (needs
an MI355X): fewer bricks than a block group, one and two wide blocks per CU,
and more bricks than the wide blocks take (256-thread blocks).  The solution
is checked by a residual formed here in FP64 from the fields read back:
||b - M p|| / ||b|| with M the 251-point operator on the dense lattice."""
import numpy as np
import pytest

from vps import Projection, scenes, _abi

pytestmark = pytest.mark.gpu


def residual(sc, f, row):
    s = sc["lattice_spacing"]
    nx, ny, nz = (int(k) for k in sc["lattice_dims"])
    H = 4 * s
    c1 = 6 / H * 8 / (np.pi * H ** 3)

    def dense(a):
        out = np.zeros(nx * ny * nz)
        out[f["node"]] = a
        return out.reshape(nz, ny, nx)

    V, p = dense(f["vol"]), dense(f["p"])
    src = np.pad(V * p if row else p, 3)
    acc = np.zeros((nz, ny, nx))
    for k in range(-3, 4):
        for j in range(-3, 4):
            for i in range(-3, 4):
                r2 = i * i + j * j + k * k
                if not 0 < r2 < 16:
                    continue
                r = np.sqrt(r2) * s
                x = r / H
                dw = c1 * (x * (3 * x - 2) if x < 0.5 else -(1 - x) ** 2)
                acc += 2 * dw / (r + 1e-6) * src[3 + k:3 + k + nz, 3 + j:3 + j + ny,
                                                 3 + i:3 + i + nx]
    acc = acc.reshape(-1)[f["node"]]
    mp = f["diag"] * f["p"] + (acc if row else f["vol"] * acc)
    # FP32 rounding of p alone (half an ulp of every entry)
    floor = 2.0 ** -24 * np.linalg.norm(f["diag"] * f["p"]) / np.linalg.norm(f["div"])
    return np.linalg.norm(f["div"] - mp) / np.linalg.norm(f["div"]), floor


# sheets: (nx, ny, nz) particles cover about (n / 8 + 1) bricks an axis
@pytest.mark.parametrize("op", [_abi.OP_TRANSPOSE, _abi.OP_ROW])
@pytest.mark.parametrize("block,lo,hi", [((5, 4, 3), 1, 8), ((121, 121, 2), 200, 320),
                                         ((133, 133, 2), 321, 512), ((170, 165, 9), 513, 3072),
                                         ((445, 445, 2), 3073, 8192)])
def test_3d_iteration_launches(block, lo, hi, op):
    dx = 1.0 / 100
    sc = scenes.dam_break(3, dx, [(b + 2) * dx for b in block], [b * dx for b in block])
    g = Projection(sc, op_mode=op)
    g.initialize()
    g.advect(5e-4, 9.8)
    for _ in range(2):
        st = g.projection_step()
        assert lo <= st["n_active_bricks"] <= hi
        assert st["cg_true_rel_residual"] < 1e-6
        r, floor = residual(sc, g.virtual(), op == _abi.OP_ROW)
        assert r < 1e-6 + 4 * floor
    g.close()
