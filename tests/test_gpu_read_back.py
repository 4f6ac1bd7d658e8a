"""Large states come back through pinned chunks on several threads: bit for bit
what was set, for sizes around the threshold and with a part chunk at the end,
and from two threads at once (one of them finds the chunks taken)."""
import threading

import numpy as np
import pytest

from vcp3d_open_amd.cases import TGVCase

pytestmark = pytest.mark.gpu


def solver(n, p, seed):
    from vcp3d_open_amd.solver import SolverClass
    s = SolverClass(TGVCase(n=n, p=p))
    u = np.random.default_rng(seed).standard_normal((s.n_elem, 5, s.n_dofs))
    s._check(s._L.vcp_set_solution(s.h, u))
    return s, u


# 17 MB and 20 MB (one chunk past the threshold and three), 30 MB, 61 MB, each with a part chunk at the end
@pytest.mark.parametrize("n,p", [(15, 4), (16, 4), (13, 6), (23, 4)])
def test_read_back(n, p):
    print(f"[case] n={n} P={p}", flush=True)
    s, u = solver(n, p, n)
    for _ in range(3):
        assert np.array_equal(s.solution(), u)


def test_read_back_from_two_threads():
    pairs = [solver(16, 4, 1), solver(17, 4, 2)]
    ok = []

    def read(s, u):
        ok.append(all(np.array_equal(s.solution(), u) for _ in range(5)))

    threads = [threading.Thread(target=read, args=pr) for pr in pairs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert ok == [True, True]
