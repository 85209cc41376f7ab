"""The PCG's launch shapes: block sizes, where the reductions are combined,
the matrix readers (ELL with 16-bit and 32-bit columns, up to 8 and up to 16
entries, CSR) and the ends of their ranges of rows.

Two checks per system, both over a fixed number of iterations (the tolerance
is never met, the cap ends the solve):
  - against the same iteration in numpy.  The matrices are diagonally dominant
    (eigenvalues of D^-1 A within [1/3, 5/3]), so twelve iterations amplify
    rounding by little: about 12 steps x 5 (condition) x 17 (terms of a row) x
    1.1e-16 = 1e-13; the bound is 1e-11;
  - up to 524,288 rows bit for bit against cfd_bicg_ex_noalloc, which reads
    the CSR arrays with blocks of 256 threads whatever the size."""
import ctypes as C

import numpy as np
import pytest

from cfd_amd.api import biCG_ex
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu

ITERS = 12


def _matrix(n, offsets, seed, shuffle=False, ragged=0):
    """Symmetric rows: diagonal first, then columns i +- o; row sums of the
    magnitudes off the diagonal at most 2/3 of it.  shuffle: a random
    renumbering (columns anywhere); ragged: the first `ragged` rows keep only
    their diagonal."""
    rng = np.random.default_rng(seed)
    i = np.arange(n)
    rows, cols, vals = [i], [i], [np.full(n, 1.5 * 2 * len(offsets) + 0.1)]
    for o in offsets:
        v = -rng.uniform(0.5, 1.0, n - o)
        a, b = i[:-o], i[o:]
        if ragged:
            v[a < ragged] = 0.0
        rows += [a, b]
        cols += [b, a]
        vals += [v, v]
    r, c, v = np.concatenate(rows), np.concatenate(cols), np.concatenate(vals)
    keep = v != 0.0
    r, c, v = r[keep], c[keep], v[keep]
    if shuffle:
        p = rng.permutation(n)
        r, c = p[r], p[c]
    order = np.lexsort((c, r != c, r))      # diagonal first in each row
    r, c, v = r[order], c[order], v[order]
    rp = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(r, minlength=n), out=rp[1:])
    diag = np.zeros(n)
    diag[r[r == c]] = v[r == c]
    fidx = (np.sort(rng.choice(n, max(1, n // 50), replace=False)) + 1).astype(np.int32)
    return dict(A=v, idx=(c + 1).astype(np.int32), rp=rp, dg=diag, n=n, r=r, c=c, fidx=fidx,
                xfix=rng.standard_normal(fidx.size), b=rng.standard_normal(n))


def _numpy_cg(sy, x0, iters):
    n = sy["n"]
    free = np.ones(n)
    free[sy["fidx"] - 1] = 0.0
    x = x0.copy()
    x[sy["fidx"] - 1] = sy["xfix"]

    def mul(p):
        return free * np.bincount(sy["r"], weights=sy["A"] * p[sy["c"]], minlength=n)
    r = free * (sy["b"] - mul(x))
    z = r / sy["dg"]
    p, e = z.copy(), r @ z
    for _ in range(iters):
        y = mul(p)
        a = e / (p @ y)
        x = x + a * p
        r = r - a * y
        z = r / sy["dg"]
        e, old = r @ z, e
        p = z + (e / old) * p
    y = mul(p)                              # the update after the last loop test
    return x + e / (p @ y) * p


NARROW, WIDE = (1, 2, 3), (1, 2, 3, 5, 7, 9, 11)


@pytest.mark.parametrize("n, offsets, shuffle, ragged", [
    (1, (), False, 0), (63, NARROW, False, 0), (257, NARROW, False, 0),
    (1025, (1, 32, 33), False, 0), (5000, NARROW, False, 3000),   # ragged: CSR
    (70000, NARROW, True, 0),                                     # 32-bit columns
    (163840, (1, 400, 401), False, 0), (163841, (1, 400, 401), False, 0),
    (262144, (1, 512, 513), False, 0), (262145, (1, 512, 513), False, 0),
    (262145, WIDE, False, 0), (300000, WIDE, True, 0),
    (524288, (1, 32767, 32768), False, 0),
])
def test_pcg_launch_shapes(n, offsets, shuffle, ragged):
    sy = _matrix(n, offsets, n, shuffle, ragged)
    sy["b"] = np.zeros(n)                   # the allocation-free test's right-hand side
    x0 = np.random.default_rng(n + 1).standard_normal(n)
    print(f"PCG on {n} rows, {sy['A'].size} entries", flush=True)
    x = x0.copy()
    it, rz, cv = biCG_ex(sy["A"], sy["idx"], sy["rp"], sy["dg"], x, sy["b"], sy["xfix"],
                         sy["fidx"], tol=1e-150, maxit=ITERS, rel=1)
    xb, itb, rzb, cvb = _noalloc(sy, x0, 1e-150, ITERS, 1)
    assert (it, cv) == (itb, cvb)
    assert np.array_equal(x.view(np.int64), xb.view(np.int64)) and (rz == rzb or n == 1)
    if n > 100:
        assert it == ITERS and not cv
        ref = _numpy_cg(sy, x0, ITERS)
        assert np.linalg.norm(x - ref) <= 1e-11 * np.linalg.norm(ref)


@pytest.mark.parametrize("n", [786432, 786433])
def test_pcg_above_the_fold(n):
    sy = _matrix(n, (1, 900, 901), n)
    x = x0 = np.random.default_rng(n + 1).standard_normal(n)
    x = x0.copy()
    print(f"PCG on {n} rows", flush=True)
    it, _, _ = biCG_ex(sy["A"], sy["idx"], sy["rp"], sy["dg"], x, sy["b"], sy["xfix"], sy["fidx"],
                       tol=1e-150, maxit=ITERS, rel=1)
    ref = _numpy_cg(sy, x0, ITERS)
    assert it == ITERS
    assert np.linalg.norm(x - ref) <= 1e-11 * np.linalg.norm(ref)


@pytest.mark.parametrize("nr", [410, 700, 1500, 2000])   # 164,410 to 802,000 rows
def test_paired_solves_meet_the_rule(nr):
    """Both mesh solves of a step in one launch per kernel (each of its block
    shapes): the residual recomputed from the solutions meets the relative
    rule r.D^-1 r <= tol^2 r0.D^-1 r0 (10 times that: the solver's own residual
    is updated, not recomputed)."""
    from scipy.sparse import csr_matrix

    from cfd_amd.mesh import ellipse_case
    from cfd_amd.solver import Session
    tol = 1e-6
    cs = ellipse_case(nr, 401)
    S = Session(cs, pcg_rel=1, pcg_tol=tol, pcg_maxit=20000)
    rp, idx = S.mesh.lap_structure()
    A = csr_matrix((S.get("LAP_SPARSE"), idx - 1, rp), shape=(cs.npoin, cs.npoin))
    diag = S.get("LAP_DIAG")
    print(f"paired solves on {cs.npoin} rows", flush=True)
    S.step(1)
    assert S.scalars()["PCG_UNCONV"] == 0 and S.scalars()["PCG_ITSUM"] > 20
    free = np.ones(cs.npoin, bool)
    free[np.asarray(cs.lists["ilaux"]) - 1] = False
    for name in ("XPOS", "YPOS"):
        x = S.get(name)
        x0 = np.where(free, 0.0, x)
        r, r0 = free * (A @ x), free * (A @ x0)
        assert np.abs(x0).max() > 0 and not np.isnan(x).any()
        assert r @ (r / diag) <= 10 * tol ** 2 * (r0 @ (r0 / diag))
