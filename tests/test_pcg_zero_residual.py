"""Mesh solves whose residual is, or becomes, exactly zero: nothing displaced, every
row fixed, a direct hit of the first step, a guess that decays to zero.  Each
path of the solver (one launch, the kernels per iteration from ELL and from CSR
rows, the one-block reductions above their limit), the allocation-free entry, and
a session whose body does not move.  Every answer is known exactly or to the
rounding of the guess; none may be a NaN."""
import numpy as np
import pytest

from cfd_amd.api import biCG_ex
from cfd_amd.mesh import ellipse_case
from cfd_amd.solver import Session
from test_pcg_shapes import _matrix
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu


def _solve(sy, x0, tol, maxit, rel):
    x = np.array(x0, np.float64)
    got = biCG_ex(sy["A"], sy["idx"], sy["rp"], sy["dg"], x, sy["b"], sy["xfix"], sy["fidx"],
                  tol=tol, maxit=maxit, rel=rel)
    return (x, *got)


def _both(sy, x0, tol, maxit, rel):
    yield _solve(sy, x0, tol, maxit, rel)
    if sy["n"] <= 524288:
        yield _noalloc(sy, x0, tol, maxit, rel)


@pytest.mark.parametrize("n, ragged", [(1, 0), (100, 0), (3500, 0), (4608, 0), (5000, 0),
                                       (5000, 3000), (262145, 0), (786433, 0)])
def test_nothing_displaced(n, ragged):
    sy = _matrix(n, (1, 30, 31) if n > 31 else (), n, ragged=ragged)
    sy["b"], sy["xfix"] = np.zeros(n), np.zeros(sy["fidx"].size)
    print(f"zero displacement on {n} rows", flush=True)
    for x, it, rz, cv in _both(sy, np.zeros(n), 1e-8, 1000, 1):
        assert (it, rz, cv) == (0, 0.0, True) and not x.any()


@pytest.mark.parametrize("n", [1, 100, 4608, 5000])
@pytest.mark.parametrize("rel", [0, 1])
def test_every_row_fixed(n, rel):
    sy = _matrix(n, (1, 30, 31) if n > 31 else (), n)
    sy["b"], sy["fidx"] = np.zeros(n), np.arange(1, n + 1, dtype=np.int32)
    sy["xfix"] = np.random.default_rng(n).standard_normal(n)
    for x, it, rz, cv in _both(sy, np.ones(n), 1e-8, 1000, rel):
        assert (it, rz, cv) == (0, 0.0, True) and np.array_equal(x, sy["xfix"])


@pytest.mark.parametrize("n", [2, 64, 4608, 5000])
def test_the_first_step_solves(n):
    """A diagonal of 4, powers of two on the right: the first step is exact."""
    sy = dict(A=np.full(n, 4.0), idx=np.arange(1, n + 1, dtype=np.int32),
              rp=np.arange(n + 1, dtype=np.int32), dg=np.full(n, 4.0), n=n, b=np.full(n, 8.0),
              fidx=np.ones(1, np.int32), xfix=np.full(1, 0.5))
    x, it, rz, cv = _solve(sy, np.zeros(n), 1e-8, 1000, 1)
    assert (it, rz, cv) == (1, 0.0, True)
    assert x[0] == 0.5 and np.all(x[1:] == 2.0)


@pytest.mark.parametrize("n", [100, 4608, 5000])
def test_a_guess_that_decays_to_zero(n):
    """The threshold is zero, the guess is not: the solve runs until its residual
    is zero or it meets the cap, and leaves the guess's rounding at most."""
    sy = _matrix(n, (1, 30, 31), n)
    sy["b"], sy["xfix"] = np.zeros(n), np.zeros(sy["fidx"].size)
    x0 = np.random.default_rng(n).standard_normal(n)
    for x, it, rz, cv in _both(sy, x0, 1e-8, 20000, 1):
        assert it > 10 and (cv or it == 20000)
        assert np.abs(x).max() <= 1e-12


@pytest.mark.parametrize("nr, nt, warm", [(24, 48, 0), (24, 48, 2), (96, 192, 0), (96, 192, 2),
                                          (420, 401, 0)])
def test_a_body_that_does_not_move(nr, nt, warm):
    """A moving-mesh session with an amplitude of zero, under the relative rule:
    the coordinates stay, the mesh velocity is zero, every solve converges."""
    cs = ellipse_case(nr, nt)
    S = Session(cs, motion=1, motion_amp=0.0, motion_omega=0.2, pcg_rel=1, pcg_tol=1e-8,
                pcg_maxit=2000, warm_start=warm)
    print(f"a resting body on {cs.npoin} nodes, warm start {warm}", flush=True)
    X, Y = S.get("X"), S.get("Y")
    S.step(5)
    assert np.array_equal(S.get("X"), X) and np.array_equal(S.get("Y"), Y)
    assert not S.get("W_X").any() and not S.get("W_Y").any()
    assert np.isfinite(S.get("U")).all()
    sc = S.scalars()
    assert sc["PCG_ITSUM"] == 0 and sc["PCG_UNCONV"] == 0
