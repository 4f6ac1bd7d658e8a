"""Faces sharing a wave (two at (4, 5), four at (3, 4)): element counts that
leave the last wave partly filled, and boxes whose block boundary leaves some
lane groups of a wave without a face, against the oracle; and the reciprocal
and root used by the pointwise fluxes over states far from the reference one
(strong jumps: the logarithmic means' closed form beside their series).

Tolerance: relative 1e-10 in the residual with each side's own metric set-up
(test_gpu_parity.py); 1e-9 on the open boxes."""
import numpy as np
import pytest

from vcp3d_open_amd.cases import OpenBoxCase, TGVCase

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


CASES = [("tgv_n2_p2", TGVCase(n=2, p=2)), ("tgv_n3_p2", TGVCase(n=3, p=2)), ("tgv_n5_p2", TGVCase(n=5, p=2, curvilinear=True)),
         ("tgv_n3_p3", TGVCase(n=3, p=3)), ("tgv_n5_p3", TGVCase(n=5, p=3, curvilinear=True)),
         ("tgv_n3_p3_rule10", TGVCase(n=3, p=3, rule=10)), ("vreman_n3_p2", TGVCase(n=3, p=2, sgs="vreman")),
         ("wale_n3_p3", TGVCase(n=3, p=3, sgs="wale")),
         ("box_p2", OpenBoxCase(n=(5, 3, 3), p=2, sponge_elems=1)), ("box_p3", OpenBoxCase(n=(7, 3, 1), p=3, sponge_elems=2))]


@pytest.mark.parametrize("bug", [True, False], ids=["bugcompat", "fixed"])
@pytest.mark.parametrize("name,case", CASES, ids=[c[0] for c in CASES])
def test_shared_waves_match_oracle(oracle_lib, name, case, bug):
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


@pytest.mark.parametrize("p", [2, 3, 4])
def test_strong_jumps_match_oracle(oracle_lib, p):
    """Element-wise constant states with density and pressure ratios up to
    30 between neighbours."""
    from vcp3d_open_amd.solver import SolverClass
    case = TGVCase(n=3, p=p)
    rng = np.random.default_rng(11 + p)
    nodal = case.initial_conservative()
    rho = nodal[..., 0].mean() * np.exp(rng.uniform(-1.7, 1.7, case.n_elems))[:, None]
    pres = case.ref["p_ref"] * np.exp(rng.uniform(-1.7, 1.7, case.n_elems))[:, None]
    vel = case.ref["u_ref"] * rng.uniform(-0.4, 0.4, (case.n_elems, 1, 3))
    nodal[..., 0] = rho
    nodal[..., 1:4] = rho[..., None] * vel
    nodal[..., 4] = pres / 0.4 + 0.5 * rho * (vel ** 2).sum(-1)
    print(f"[case] strong jumps P={p}", flush=True)
    o, g = oracle_lib.Oracle(case), SolverClass(case)
    o.set_restart(nodal)
    g.ReadRestartSolution(nodal)
    o.residual()
    g.Residual(True)
    assert rel(g.residual_array(), o.residual_array()) < 1e-10
