"""The column form of the volume kernel (one thread per column of points)
against the workgroup form and the oracle, at element counts around its
workgroups' edges: shapes that put four and two elements into a wave with the
last workgroup partly filled, one element per wave, and columns split over the
halves of a workgroup (K >= 6 in FP64), with an SGS model, a sponge with
matching layer and a body force (the kernel's full form).

Tolerances: the residual's conditioning turns summation-order differences of
1e-16 into 1e-12 .. 1e-11 (test_gpu_parity.py: 3e-11 on shared geometry); one
iteration more or less of the solve changes it by the stop rule's 1e-10. States
after steps agree to rounding (1e-14). The float form stops its solve at 1e-5
and carries 6e-8 rounding, amplified in the residual by the cancellation of
the pressure fluxes: 2e-3 in the residual, 1e-6 in the state (test_gpu_mixed.py).
"""
import numpy as np
import pytest

from vcp3d_open_amd.cases import OpenBoxCase, TGVCase

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def cases():
    out = []
    for p, rule in ((2, None), (3, None), (3, 10), (4, None), (5, None), (6, None)):
        for n in (2, 3):          # 8 and 27 elements: full and partly filled workgroups
            out.append((f"tgv_n{n}_p{p}_rule{rule}", TGVCase(n=n, p=p, rule=rule, mach=0.3, phase=(0.2, 0.9, 0.4))))
        out.append((f"curv_n4_p{p}_rule{rule}", TGVCase(n=4, p=p, rule=rule, curvilinear=True)))
    out.append(("wale_p2", TGVCase(n=3, p=2, sgs="wale")))
    out.append(("vreman_p5", TGVCase(n=3, p=5, sgs="vreman")))
    out.append(("body_force_p3", TGVCase(n=3, p=3, body_force=(3000.0, -1500.0, 800.0))))
    for p in (2, 4, 6):           # 5 x 3 x 3 elements: one partly filled workgroup
        out.append((f"box_p{p}", OpenBoxCase(n=(5, 3, 3), p=p, sponge_elems=2)))
    return out


def evaluate(case, tile, bug, precision):
    from vcp3d_open_amd.solver import SolverClass
    g = SolverClass(case, bug_compat=bug, precision=precision)
    g.set_tile(tile)
    g.ReadRestartSolution(case.initial_conservative())
    if isinstance(case, OpenBoxCase):
        g.SetDampingState(case.damping_primitive())
    mon = g.Residual(True)
    res, iters = g.residual_array(), g.cg_iterations()
    for _ in range(2):
        g.ExecuteTimeSynchronizationStep()
    return res, iters, g.solution(), mon


@pytest.mark.parametrize("bug", [True, False], ids=["bugcompat", "fixed"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("name,case", cases(), ids=[c[0] for c in cases()])
def test_columns_match_workgroups(name, case, precision, bug):
    from vcp3d_open_amd.solver import volume_tiles
    print(f"[case] {name} {precision} bug={bug}", flush=True)
    tiles = volume_tiles(case.p + 1, case.rule // 2 + 1)
    a = evaluate(case, tiles[0], bug, precision)
    b = evaluate(case, tiles[1] if len(tiles) > 1 else 0, bug, precision)
    tol_r, tol_u = (3e-10, 1e-14) if precision == "fp64" else (2e-3, 1e-6)
    assert rel(a[0], b[0]) < tol_r
    assert rel(a[2], b[2]) < tol_u
    assert np.abs(a[1] - b[1]).max() <= 1
    scale = np.abs(b[3]).max()
    assert np.abs(a[3] - b[3]).max() <= (1e-11 if precision == "fp64" else 1e-5) * scale


def test_default_follows_the_element_count():
    """The default is the column kernel for a large case and the workgroup
    kernel for a small one, bit for bit."""
    from vcp3d_open_amd.solver import volume_tiles
    for n, which in ((6, 1), (11, 0)):
        case = TGVCase(n=n, p=3)
        tiles = volume_tiles(4, 5)
        d = evaluate(case, 0, True, "fp64")
        t = evaluate(case, tiles[which], True, "fp64")
        assert np.array_equal(d[2], t[2]) and np.array_equal(d[0], t[0])


def test_batch_takes_the_same_kernels():
    """Cases of one (K, M) that take different volume kernels (by size and by
    their terms) share a batch and each matches itself in a batch of one."""
    from vcp3d_open_amd.solver import Batch, SolverClass
    members = [TGVCase(n=3, p=3), TGVCase(n=11, p=3, mach=0.2), OpenBoxCase(n=(6, 2, 2), p=3, sponge_elems=2),
               OpenBoxCase(n=(18, 8, 8), p=3, sponge_elems=3), TGVCase(n=11, p=3, sgs="wale")]

    def make(c):
        g = SolverClass(c)
        g.ReadRestartSolution(c.initial_conservative())
        if isinstance(c, OpenBoxCase):
            g.SetDampingState(c.damping_primitive())
        return g

    together = [make(c) for c in members]
    batch = Batch()
    for g in together:
        batch.add(g, 3)
    batch.step(3)
    batch.wait()
    for c, g in zip(members, together):
        one = make(c)
        b = Batch()
        b.add(one, 3)
        b.step(3)
        b.wait()
        assert np.array_equal(g.solution(), one.solution())
        b.close()
