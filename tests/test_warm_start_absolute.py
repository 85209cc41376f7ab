"""The learned start under the absolute rule: a step after one whose two solves both made
no iteration skips the learned candidate.  Small meshes, whose solves run in one
launch and are asked for their iterations without waiting, against the same solves
by the kernels per iteration (an iteration cap above the one launch's), whose polls
tell; in one call of many steps, step by step, and after the run is begun again."""
import numpy as np
import pytest

from cfd_amd.mesh import ellipse_case
from cfd_amd.solver import Session

pytestmark = pytest.mark.gpu

FIELDS = ("U", "X", "Y", "XPOS", "YPOS", "W_X")
COUNTS = ("PCG_ITSUM", "PCG_UNCONV", "WS_LEARNED", "WS_SOLVES", "WS_LOSS")


def _run(warm, amp, maxit, calls, again=False):
    cs = ellipse_case(24, 48)
    S = Session(cs, motion=1, motion_amp=amp, motion_omega=0.2, pcg_tol=1e-10, pcg_maxit=maxit,
                warm_start=warm)
    if again:                               # on the mesh as it stands
        S.step(7)
        S.init_freestream()
    base = S.scalars()
    for n in calls:
        S.step(n)
    sc = S.scalars()
    return [S.get(f).tobytes() for f in FIELDS], [sc[k] - (base[k] if "SUM" in k or "SOLVES" in k
                                                           or "LEARNED" in k else 0.0) for k in COUNTS]


@pytest.mark.parametrize("warm", [1, 2])
@pytest.mark.parametrize("amp", [1e-6, 1e-2, 0.3])   # no iterations, some steps with, all with
def test_asked_and_polled_solves_agree(warm, amp):
    print(f"warm start {warm}, amplitude {amp:g}", flush=True)
    f, c = _run(warm, amp, 1000, [12])
    fp, cp = _run(warm, amp, 20001, [12])
    assert f == fp and c == cp
    assert _run(warm, amp, 1000, [1] * 12) == (f, c)
    assert _run(warm, amp, 1000, [5, 7]) == (f, c)
    print("iterations, unconverged, learned, solves, loss:", c)


def test_after_the_run_is_begun_again():
    assert _run(2, 1e-2, 1000, [6], again=True) == _run(2, 1e-2, 20001, [6], again=True)
