"""The 2D iteration limit holds where a residual replacement falls on it (needs an
MI355X): a solve that converged on its recursion in the last iteration allowed,
but not on the true residual, stops there.  CG on the rows as written replaces
about once a solve from a zero start, so every limit around a solve's own
iterations is tried; the solve of that limit reports at most as many."""
import pytest

from vps import Projection, _abi, scenes

pytestmark = pytest.mark.gpu


def test_limit_at_a_replacement():
    on_limit = 0
    for seed in range(1, 13):
        sc = scenes.small_2d(20, seed=seed)

        def solve(limit):
            g = Projection(sc, op_mode=_abi.OP_ROW, warm_start=_abi.WARM_ZERO,
                           max_iterations=limit)
            g.initialize()
            g.advect(1e-3, 9.8)
            g.refresh_real()
            g.generate_particles()
            s = g.project(allow_fail=True)
            g.close()
            return s

        free = solve(-1)
        assert free["status"] == 0
        for limit in range(max(1, free["cg_iterations"] - 6), free["cg_iterations"] + 1):
            s = solve(limit)
            assert s["cg_iterations"] <= limit, (seed, limit)
            if s["status"] == 0:
                assert s["cg_true_rel_residual"] < 1e-6
            else:
                on_limit += s["cg_iterations"] == limit
    assert on_limit > 0
