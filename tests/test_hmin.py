"""The smallest element of a moving mesh (HMIN), folded by a block of laplace's launch
from the partials that deriv left: against the minimum of HH, from a handful of
partials to more than a wave's lanes take in one batch of sixteen loads each."""
import numpy as np
import pytest

from cfd_amd.mesh import ellipse_case
from cfd_amd.solver import Session

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr, nt", [(6, 12), (33, 65), (97, 193), (385, 701), (1000, 2049)])
@pytest.mark.parametrize("gcl", [-1, 1])
def test_hmin_is_the_smallest_hh(nr, nt, gcl):
    cs = ellipse_case(nr, nt)
    S = Session(cs, gcl=gcl, motion=1, motion_amp=0.05, motion_omega=0.2)
    print(f"HMIN of {cs.nelem} triangles", flush=True)
    for _ in range(2):
        assert S.scalars()["HMIN"] == min(S.get("HH").min(), 1.0e10)
        S.step(1)
    assert np.isfinite(S.get("X")).all()
