"""Solves of a caller's matrix begin on its CSR rows and go on with a copy in ELL order
once they have proved long (28 iterations up to 131,072 rows, 108 above; small ones
after the first test): every row reader and block size on that copy, the change
over itself at each of its edges, and iterations that are queued ahead, bit for bit
against cfd_bicg_ex_noalloc, which stays on the CSR rows; above its size against the
iteration in numpy (converged by then: bound as in test_pcg_shapes)."""
import numpy as np
import pytest

from cfd_amd.api import biCG_ex
from test_pcg_shapes import NARROW, WIDE, _matrix, _numpy_cg
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu


def _long(sy, x0, maxit, tol=1e-150):
    x = x0.copy()
    return (x, *biCG_ex(sy["A"], sy["idx"], sy["rp"], sy["dg"], x, sy["b"], sy["xfix"], sy["fidx"],
                        tol=tol, maxit=maxit, rel=1))


@pytest.mark.parametrize("n, offsets, shuffle, ragged, caps", [
    (4864, (1, 30, 31), False, 0, (0, 1, 40)), (4865, (1, 30, 31), False, 0, (27, 28, 29, 30, 31, 140)),
    (5000, NARROW, False, 3000, (28, 29, 140)),                   # no copy: ragged
    (3000, WIDE, False, 0, (0, 28, 29, 140)),                     # small, but rows of 15
    (70000, NARROW, True, 0, (28, 31, 140)),                      # 32-bit columns
    (131072, (1, 400, 401), False, 0, (29, 140)), (131073, (1, 400, 401), False, 0, (108, 109, 140)),
    (163840, (1, 400, 401), False, 0, (140,)), (163841, (1, 400, 401), False, 0, (140,)),
    (262144, (1, 512, 513), False, 0, (140,)), (262145, (1, 512, 513), False, 0, (107, 108, 110, 140)),
    (262145, WIDE, False, 0, (140,)), (300000, WIDE, True, 0, (140,)),
    (524288, (1, 32767, 32768), False, 0, (140,)),
])
def test_the_copy_goes_on_where_the_rows_stand(n, offsets, shuffle, ragged, caps):
    sy = _matrix(n, offsets, n, shuffle, ragged)
    sy["b"] = np.zeros(n)                   # the allocation-free test's right-hand side
    x0 = np.random.default_rng(n + 1).standard_normal(n)
    for cap in caps:
        print(f"PCG on {n} rows, {cap} iterations", flush=True)
        x, it, rz, cv = _long(sy, x0, cap)
        xb, itb, rzb, cvb = _noalloc(sy, x0, 1e-150, cap, 1)
        assert (it, rz, cv) == (itb, rzb, cvb) and it == cap
        assert np.array_equal(x.view(np.int64), xb.view(np.int64))


@pytest.mark.parametrize("n", [786432, 786433])
def test_above_the_fold(n):
    sy = _matrix(n, (1, 900, 901), n)
    x0 = np.random.default_rng(n + 1).standard_normal(n)
    print(f"PCG on {n} rows", flush=True)
    x, it, _, _ = _long(sy, x0, 120)
    ref = _numpy_cg(sy, x0, 120)
    assert it == 120 and np.linalg.norm(x - ref) <= 1e-11 * np.linalg.norm(ref)
