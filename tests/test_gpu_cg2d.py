"""The one-launch 2D CG iteration against the FP64 oracle (needs an MI355X):
one brick row (fewer bricks than a block holds), ragged brick counts, and a
lattice with more bricks than one pass of the largest grid covers (the
grid-strided rounds), for both operators.  Bars as in the parity tests; the
iteration count is compared for the default operator only (CG on the rows as
written converges slowly and unevenly near the tolerance)."""
import numpy as np
import pytest

import oracle_py as O
from vps import Projection, scenes, _abi

pytestmark = pytest.mark.gpu


# bricks of 8 x 8 nodes; a block holds four, a grid at most three per CU
@pytest.mark.parametrize("op", [_abi.OP_TRANSPOSE, _abi.OP_ROW])
@pytest.mark.parametrize("block,box", [((4, 4), (8, 8)), ((9, 5), (17, 11)),
                                       ((31, 44), (60, 50)), ((520, 430), (524, 434))])
def test_2d_iteration(block, box, op):
    dx = 1.0 / max(box)
    sc = scenes.dam_break(2, dx, [b * dx for b in box], [b * dx for b in block])
    kw = dict(op_mode=op)
    o = O.Oracle(sc, **kw)
    o.initialize()
    g = Projection(sc, **kw)
    g.initialize()
    for step in range(2):
        o.advect(1e-4, 9.8)
        g.advect(1e-4, 9.8)
        so = o.projection_step()
        sg = g.projection_step()
        if op == _abi.OP_TRANSPOSE:
            assert abs(sg["cg_iterations"] - so["cg_iterations"]) <= 1, step
        assert sg["cg_true_rel_residual"] < 1e-6, step
        vo, vg = o.virtual(), g.virtual()
        assert np.array_equal(vo["node"], vg["node"]), step
        assert np.linalg.norm(vg["p"] - vo["p"]) / np.linalg.norm(vo["p"]) < 1e-4, step
        v_o, v_g = o.particles()[1], g.particles()[1]
        assert np.linalg.norm(v_g - v_o) / np.linalg.norm(v_o) < 1e-4, step
    g.close()
