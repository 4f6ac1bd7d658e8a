"""Faces of two waves (M = 9) and the odd line pitches of even M: residual,
monitored maxima and the eddy viscosity's maximum over both waves against the
oracle, for element counts down to the smallest box.

Tolerance: relative 1e-10 in the residual with each side's own metric set-up
(test_gpu_parity.py), 1e-9 on the open boxes; the eddy-viscosity maximum 1e-9
(test_gpu_sgs.py)."""
import numpy as np
import pytest

from vcp3d_open_amd.cases import OpenBoxCase, TGVCase

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


CASES = [("tgv_n2_p6", TGVCase(n=2, p=6)), ("tgv_n3_p6", TGVCase(n=3, p=6)),
         ("tgv_n4_p6", TGVCase(n=4, p=6, curvilinear=True)), ("wale_n3_p6", TGVCase(n=3, p=6, sgs="wale")),
         ("vreman_n4_p6", TGVCase(n=4, p=6, sgs="vreman", curvilinear=True)),
         ("box_p6", OpenBoxCase(n=(5, 3, 1), p=6, sponge_elems=1)),
         ("tgv_n3_p5", TGVCase(n=3, p=5)), ("tgv_n3_p3_rule10", TGVCase(n=3, p=3, rule=10))]


@pytest.mark.parametrize("bug", [True, False], ids=["bugcompat", "fixed"])
@pytest.mark.parametrize("name,case", CASES, ids=[c[0] for c in CASES])
def test_faces_match_oracle(oracle_lib, name, case, bug):
    from vcp3d_open_amd.solver import SolverClass
    print(f"[case] {name} bug={bug}", flush=True)
    o = oracle_lib.Oracle(case, bug_compat=bug)
    g = SolverClass(case, bug_compat=bug)
    nodal = case.initial_conservative()
    o.set_restart(nodal)
    g.ReadRestartSolution(nodal)
    box = isinstance(case, OpenBoxCase)
    if box:
        o.set_damping_state(case.damping_primitive())
        g.SetDampingState(case.damping_primitive())
    md_o = o.residual()
    md_g = g.Residual(True)
    assert rel(g.residual_array(), o.residual_array()) < (1e-9 if box else 1e-10)
    assert abs(md_g[6] - md_o[6]) <= 1e-9 * md_o[6]
    if getattr(case, "sgs", "none") != "none":
        assert md_o[7] > 0.0
        assert abs(md_g[7] - md_o[7]) <= 1e-9 * md_o[7]
