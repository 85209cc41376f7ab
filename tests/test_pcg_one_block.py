"""The PCG of small systems, a whole solve in one launch: the ends of each of
its shapes (rows per thread, values in registers, LDS and memory, 7 and 8
entries a row), bit for bit against cfd_bicg_ex_noalloc (the kernels per
iteration, CSR rows) on the solution, the iterations, the final r.z and the
outcome: an iteration cap, the first test, a tolerance met, no fixed nodes'
change."""
import numpy as np
import pytest

from cfd_amd.api import biCG_ex
from test_pcg_shapes import _matrix
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu

SEVEN, EIGHT = (1, 30, 31), (1, 2, 30, 31)


def _both(sy, x0, tol, maxit, rel):
    x = x0.copy()
    got = biCG_ex(sy["A"], sy["idx"], sy["rp"], sy["dg"], x, sy["b"], sy["xfix"], sy["fidx"],
                  tol=tol, maxit=maxit, rel=rel)
    xb, it, rz, cv = _noalloc(sy, x0, tol, maxit, rel)
    assert np.array_equal(x.view(np.int64), xb.view(np.int64))
    assert (got[0], got[2]) == (it, cv) and got[1] == rz
    return it, cv


@pytest.mark.parametrize("n", [100, 255, 512, 1023, 1024, 1025, 2048, 2049, 3071, 3073, 3500,
                               4096, 4097, 4608, 4863, 4864, 4865])
@pytest.mark.parametrize("offsets", [SEVEN, EIGHT])
def test_one_block_solves(n, offsets):
    sy = _matrix(n, offsets, n)
    if offsets is EIGHT:                    # of the pairs (i, i + 2) one a row: eight entries
        lo, far = np.minimum(sy["r"], sy["c"]), np.abs(sy["r"] - sy["c"])
        keep = (far != 2) | (lo % 4 < 2)
        sy["A"], sy["idx"], sy["r"], sy["c"] = (sy[k][keep] for k in ("A", "idx", "r", "c"))
        sy["rp"][1:] = np.cumsum(np.bincount(sy["r"], minlength=n))
    sy["b"] = np.zeros(n)                   # the allocation-free test's right-hand side
    assert np.diff(sy["rp"]).max() == (8 if offsets is EIGHT else 7)
    x0 = np.random.default_rng(n + 1).standard_normal(n)
    print(f"one-block PCG on {n} rows", flush=True)
    assert _both(sy, x0, 1e-150, 12, 1) == (12, 0)      # the cap
    assert _both(sy, x0, 1e-150, 0, 0)[0] == 0
    it, cv = _both(sy, x0, 1e-10, 1000, 1)              # relative, met
    assert cv and it > 3
    it, cv = _both(sy, x0, 1e-10, 1000, 0)              # absolute, met
    assert cv and it > 3
    assert _both(sy, x0, 1e30, 1000, 0) == (0, 1)       # the first test ends it


def test_caps_that_the_launch_leaves_to_the_loop():
    """A cap above the one launch's takes the kernels per iteration: the same
    result as a cap below it that is not reached."""
    sy = _matrix(2000, SEVEN, 7)
    x0 = np.random.default_rng(8).standard_normal(2000)
    out = []
    for maxit in (20000, 20001):
        x = x0.copy()
        r = biCG_ex(sy["A"], sy["idx"], sy["rp"], sy["dg"], x, sy["b"], sy["xfix"], sy["fidx"],
                    tol=1e-12, maxit=maxit, rel=1)
        out.append((r, x.tobytes()))
    assert out[0] == out[1]
