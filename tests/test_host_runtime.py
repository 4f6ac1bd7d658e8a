"""Host code of the library (contexts, batches, readbacks) on a stand-in for the
HIP runtime (hip_host.cpp): no GPU, kernels recorded and not run. Each test is a
process of its own, so that the stand-in never meets the real runtime."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, sys
import numpy as np
rt = ctypes.CDLL({lib!r}, mode=ctypes.RTLD_GLOBAL)
rt.rt_launches.restype = ctypes.c_char_p
rt.rt_fail_new.argtypes = [ctypes.c_long]
from vcp3d_open_amd.cases import OpenBoxCase, TGVCase
from vcp3d_open_amd.solver import Batch, SolverClass, VCPError

def launches(kernel):
    return [line for line in rt.rt_launches().decode().splitlines() if kernel in line]

def solver(precision="fp64", **kw):
    s = SolverClass(TGVCase(**kw), precision=precision)
    s.ReadRestartSolution(TGVCase(**kw).initial_conservative())
    return s
"""


@pytest.fixture(scope="session")
def host_runtime(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("hip_host") / "libhip_host.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-o", lib, os.path.join(HERE, "hip_host.cpp")],
                   check=True)

    def run(script):
        p = subprocess.run([sys.executable, "-c", PRELUDE.format(lib=lib) + script], cwd=ROOT, capture_output=True,
                           text=True, timeout=120)
        assert p.returncode == 0, f"exit {p.returncode}\n{p.stdout}\n{p.stderr}"
        return p.stdout

    return run


def test_batch_whose_group_was_emptied(host_runtime):
    """A group that has lost its last case launches nothing: not in a profile,
    which visits every group, and not in a step."""
    host_runtime("""
a, b = solver(n=3, p=2), solver(n=3, p=3)
batch = Batch()
batch.add(a); batch.add(b)
batch.step(1); batch.wait()
batch.remove(a)
rt.rt_clear()
assert len(batch.profile(1)) == 2
assert not launches("_kernel<3,")
assert len(launches("volume")) == 1
batch.step(1); batch.wait()
assert not launches("_kernel<3,")
""")


# 1.1 KB (a kernel's stores), 1.1 MB (one copy) and 18 MB (chunks on several threads)
@pytest.mark.parametrize("n,p", [(2, 2), (6, 4), (15, 4)])
def test_read_back_on_another_current_device(host_runtime, n, p):
    """A host thread whose current device is not the context's reads its
    states, as it sets them, and keeps its current device."""
    host_runtime(f"""
s = solver(n={n}, p={p})
u = np.random.default_rng(1).standard_normal((s.n_elem, 5, s.n_dofs))
rt.rt_set_device(1)
s.set_solution(u)
assert np.array_equal(s.solution(), u)
s.residual_array()
assert rt.rt_device() == 1
""")


def test_staged_read_back_without_memory_for_its_threads(host_runtime):
    """An allocation that fails anywhere in a staged readback, also while its
    threads are being started, is an error of that call or none at all; the
    process goes on and the next readback is whole."""
    host_runtime("""
s = solver(n=15, p=4)
u = np.random.default_rng(1).standard_normal((s.n_elem, 5, s.n_dofs))
s.set_solution(u)
out = np.zeros_like(u)
for after in range(14):
    out[:] = 0.0
    rt.rt_fail_new(after)
    rc = s._L.vcp_get_solution(s.h, out)
    rt.rt_fail_new(-1)
    assert rc < 0 or np.array_equal(out, u)
    assert np.array_equal(s.solution(), u)
""")


def test_cases_joining_a_batch_share_their_first_launches(host_runtime):
    """The first residual of the cases that join a batch takes one volume launch
    per kernel among them, however many they are."""
    host_runtime("""
batch = Batch()
running = solver(n=3, p=3)
batch.add(running)
batch.step(1)
late = [solver(n=3, p=3), solver(n=11, p=3), solver(n=4, p=3)]
for s in late:
    batch.add(s)
rt.rt_clear()
batch.step(0)
elements = sorted(int(line.split()[-1]) for line in launches("volume"))
# (4, 5): one workgroup per element of the small cases, one of the column kernel per two of the large one
assert elements == [27 + 64, (1331 + 1) // 2], launches("volume")
assert len(launches("face")) == 1
""")


TGV, BOX = "TGVCase(n={})", "OpenBoxCase(n=({}, 8, 8), sponge_elems=2)"


# elements, and whether they take the column kernel: both sides of each line
@pytest.mark.parametrize("precision,p,case,size,columns", [
    ("fp64", 3, TGV, 10, False), ("fp64", 3, TGV, 11, True), ("fp64", 4, TGV, 9, False), ("fp64", 4, TGV, 10, True),
    ("fp64", 5, TGV, 3, True), ("fp64", 6, TGV, 6, False), ("fp64", 6, TGV, 7, True),
    ("mixed", 3, TGV, 11, False), ("mixed", 3, TGV, 12, True), ("mixed", 4, TGV, 9, False), ("mixed", 4, TGV, 10, True),
    ("mixed", 5, TGV, 9, False), ("mixed", 5, TGV, 10, True), ("mixed", 6, TGV, 8, False), ("mixed", 6, TGV, 9, True),
    ("fp64", 3, BOX, 40, False), ("fp64", 3, BOX, 41, True), ("fp64", 4, BOX, 48, False), ("fp64", 4, BOX, 49, True),
    ("mixed", 3, BOX, 48, False), ("mixed", 3, BOX, 49, True), ("mixed", 4, BOX, 24, False), ("mixed", 4, BOX, 25, True),
    ("mixed", 5, BOX, 36, False), ("mixed", 5, BOX, 37, True)])
def test_volume_kernel_by_element_count(host_runtime, precision, p, case, size, columns):
    case = case.format(size)[:-1] + f", p={p})"
    host_runtime(f"""
case = {case}
s = SolverClass(case, precision={precision!r})
s.ReadRestartSolution(case.initial_conservative())
if isinstance(case, OpenBoxCase):
    s.SetDampingState(case.damping_primitive())
rt.rt_clear()
s.Residual(False)
taken, = launches("volume")
assert taken.startswith("volume_cols_kernel<") == {columns}, taken
# in mixed precision the faces follow: their flux lifted in double beside the column kernel
if {precision!r} == "mixed":
    face, = launches("face_kernel")
    assert ("float, double" in face) == {columns}, face
""")


def test_groups_report_the_kernel_that_runs(host_runtime):
    """A group's volume size is the one that runs: the given one, the one that
    all its cases take by themselves, or 0 where none names it (cases that differ,
    the split columns of P = 2)."""
    host_runtime("""
small, large, low = solver(n=3, p=4), solver(n=10, p=4), solver(n=3, p=2)
batch = Batch()
size = lambda K: next(g["nt"] for g in batch.groups() if g["K"] == K)
batch.add(small); batch.add(low)
assert size(5) == 256 and size(3) == 0
batch.add(large)
assert size(5) == 0
batch.remove(small)
assert size(5) == 64
batch.set_tile(5, 7, 512)
assert size(5) == 512
batch.set_tile(5, 7, 0)
batch.step(1)
assert [line for line in launches("volume") if "<5, 7, 512" in line] == []
""")
