"""Column kernel with the columns in halves of a wave (P = 2, up to 4096
elements): element counts that leave the last wave half empty and both sides of
the rule's line, in the plain form and with a subgrid model, a sponge with
matching layer and a body force, against the oracle; and the float form against
the whole-column kernel (the largest workgroup named by its tile).

Tolerance: relative 1e-10 in the residual with each side's own metric set-up
(test_gpu_parity.py), 1e-9 on the open boxes; 4e-3 between two float forms, each
within 2e-3 of FP64 (test_gpu_mixed.py)."""
import numpy as np
import pytest

from vcp3d_open_amd.cases import OpenBoxCase, TGVCase

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


CASES = [("n2", TGVCase(n=2, p=2)), ("n3", TGVCase(n=3, p=2)), ("n5_curv", TGVCase(n=5, p=2, curvilinear=True)),
         ("n16", TGVCase(n=16, p=2)), ("n17", TGVCase(n=17, p=2)),
         ("wale", TGVCase(n=3, p=2, sgs="wale")), ("vreman", TGVCase(n=5, p=2, sgs="vreman")),
         ("force", TGVCase(n=3, p=2, body_force=(3000.0, -1500.0, 800.0))),
         ("box", OpenBoxCase(n=(5, 3, 3), p=2, sponge_elems=2))]


@pytest.mark.parametrize("bug", [True, False], ids=["bugcompat", "fixed"])
@pytest.mark.parametrize("name,case", CASES, ids=[c[0] for c in CASES])
def test_halves_match_oracle(oracle_lib, name, case, bug):
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
    o.residual()
    g.Residual(True)
    assert rel(g.residual_array(), o.residual_array()) < (1e-9 if box else 1e-10)


@pytest.mark.parametrize("n", [3, 16])
def test_float_halves_match_whole_columns(n):
    from vcp3d_open_amd.solver import SolverClass
    case = TGVCase(n=n, p=2)
    print(f"[case] float n={n}", flush=True)
    out = []
    for tile in (0, 16):
        g = SolverClass(case, precision="mixed")
        g.set_tile(tile)
        g.ReadRestartSolution(case.initial_conservative())
        g.Residual(True)
        out.append(g.residual_array())
    assert rel(out[0], out[1]) < 4e-3
