"""The 2D solve stops where the caller's tolerance says (needs an MI355X).

Without the FP64 check the iterations are the oracle's: at loose tolerances the
FP32 recursion's residual agrees with it to about 1e-6, far less than an
iteration's gain.

CG on the rows as written falls unevenly and levels off near the tolerance: a
stricter threshold costs it tens of iterations, or the solve.  Over many small
scenes every solve converges, in the oracle's iterations on average; a residual
replacement (about one a solve here) adds two to four of about sixty, so
within 8%."""
import pytest

import oracle_py as O
from vps import Projection, _abi, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tolerance", [0.5, 0.3, 0.2, 0.1, 0.07, 0.04, 0.02, 0.01, 5e-3, 2e-3])
def test_unchecked_iterations(tolerance):
    sc = scenes.small_2d(20)
    o, g = O.Oracle(sc, tolerance=tolerance), Projection(sc, tolerance=tolerance)
    o.initialize()
    g.initialize()
    g.set_check_true_residual(False)
    for _ in range(4):
        o.advect(1e-3, 9.8)
        g.advect(1e-3, 9.8)
        assert g.projection_step()["cg_iterations"] == o.projection_step()["cg_iterations"]
    g.close()
    o.close()


@pytest.mark.parametrize("viscosity", [0.01, 0.0])
def test_row_operator_iterations(viscosity):
    kw = dict(op_mode=_abi.OP_ROW, warm_start=_abi.WARM_ZERO)
    its = [0, 0]
    for seed in range(1, 25):
        sc = scenes.small_2d(20 if seed % 2 else 30, seed=seed)
        for i, cls in enumerate((O.Oracle, Projection)):
            c = cls(sc, **kw)
            c.initialize()
            for _ in range(6):
                its[i] += c.advance(1e-3, 9.8, viscosity, scenes.box_colliders(sc),
                                    True)["cg_iterations"]
            c.close()
    assert its[1] <= 1.08 * its[0]
