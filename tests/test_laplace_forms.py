"""laplace's three forms give the same matrix bit for bit: the host entry (weights formed
from the coordinates in the same launch), a session's with the masses, and one with
the geometric conservation law (weights from deriv), at set-up and after steps, with
rows of up to 18 entries."""
import numpy as np
import pytest

from cfd_amd.api import MeshContext
from cfd_amd.mesh import ellipse_case
from cfd_amd.solver import Session
from test_csr_sessions import _with_star

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr, nt", [(3, 7), (8, 8), (24, 48), (131, 257)])
@pytest.mark.parametrize("star", [False, True])
@pytest.mark.parametrize("moving, gcl", [(0, -1), (1, -1), (1, 0), (1, 1)])
def test_one_matrix(nr, nt, star, moving, gcl):
    cs = ellipse_case(nr, nt, moving=moving)
    if star:
        cs = _with_star(cs)
    S = Session(cs, motion=1, motion_amp=0.01, motion_omega=0.2, gcl=gcl)
    mc = MeshContext(cs.mesh.inpoel, cs.npoin)
    for steps in (0, 2):
        S.step(steps)
        lap, diag = mc.laplace(S.get("X"), S.get("Y"), S.get("DNX"), S.get("DNY"))
        assert np.isfinite(lap).all()
        assert np.array_equal(lap, S.get("LAP_SPARSE")) and np.array_equal(diag, S.get("LAP_DIAG"))
