"""Threads with problems of different sizes at once: the one-block mesh solves and
the node-order smoothing ask for an amount of LDS that goes with the size, and a
kernel's limit of it holds for the whole process.  Each thread gets bit for bit
what the same calls give one after the other."""
import threading

import numpy as np
import pytest

from cfd_amd.api import MeshContext, biCG_ex
from cfd_amd.mesh import cylinder_case
from test_pcg_shapes import _matrix

pytestmark = pytest.mark.gpu

SOLVES = (3100, 3600, 4090, 4200, 4608, 4864)      # beside p 3 values a row in LDS, x and 2
MESHES = ((34, 96), (60, 100), (70, 130), (96, 98))


def _solve(n):
    sy = _matrix(n, (1, 30, 31), n)
    x = np.random.default_rng(n).standard_normal(n)

    def run():
        y = x.copy()
        r = biCG_ex(sy["A"], sy["idx"], sy["rp"], sy["dg"], y, sy["b"], sy["xfix"], sy["fidx"],
                    tol=1e-10, maxit=1000, rel=1)
        return r, y.tobytes()
    return run


def _smooth(nr, nt):
    m = cylinder_case(nr, nt).mesh
    fixed = np.zeros(m.npoin, np.int32)
    fixed[: m.nt] = fixed[-m.nt:] = 1
    mc = MeshContext(m.inpoel, m.npoin)

    def run():
        x, y, n, h = mc.smoothing(m.x, m.y, fixed)
        return n, h, x.tobytes(), y.tobytes()
    return run


@pytest.mark.parametrize("jobs", [[(_solve, (n,)) for n in SOLVES], [(_smooth, a) for a in MESHES]],
                         ids=["solves", "smoothing"])
def test_sizes_side_by_side(jobs):
    runs = [make(*a) for make, a in jobs]
    alone = [run() for run in runs]
    print(f"{len(runs)} threads", flush=True)
    got = [[] for _ in runs]
    start = threading.Barrier(len(runs))

    def work(k):
        start.wait()
        try:
            for _ in range(8):
                got[k].append(runs[k]())
        except Exception as e:  # noqa: BLE001 - shown below
            got[k].append(e)
    th = [threading.Thread(target=work, args=(k,)) for k in range(len(runs))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for k, a in enumerate(alone):
        assert all(g == a for g in got[k]) and len(got[k]) == 8, got[k][-1] if got[k] else None
