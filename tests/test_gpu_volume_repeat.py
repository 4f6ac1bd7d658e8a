"""Repeated residuals of the column volume kernel over elements of two and more
waves are bit-identical: the waves of an element exchange the solve's vectors
through LDS in every iteration, so a wave that reads before the other's stores
have arrived shows up as a difference (or as a solve that does not converge).
More elements than the chip holds at once, so that the waves of later ones
start at different times."""
import numpy as np
import pytest

from vcp3d_open_amd.cases import TGVCase

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,p", [(12, 5), (10, 6)])
def test_repeated_residuals_are_identical(n, p, precision):
    from vcp3d_open_amd.solver import SolverClass
    case = TGVCase(n=n, p=p)
    print(f"[case] n={n} P={p} {precision}", flush=True)
    g = SolverClass(case, precision=precision)
    g.ReadRestartSolution(case.initial_conservative())
    g.Residual(False)
    first, iters = g.residual_array(), g.cg_iterations()
    for _ in range(20):
        g.Residual(False)
        assert np.array_equal(g.residual_array(), first)
        assert np.array_equal(g.cg_iterations(), iters)
