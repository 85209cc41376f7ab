"""Moving meshes: several steps of one call against the same steps called one by one,
bit for bit in every field and scalar: element terms, areas and W of the step
before, forces beside TRANSF (up to 512 edges), the smallest element, the few-patch
forms, with and without the geometric conservation law, and with set-up calls
(reads of fields and scalars) between the calls."""
import numpy as np
import pytest

from cfd_amd.mesh import ellipse_case
from cfd_amd.solver import Session

pytestmark = pytest.mark.gpu

FIELDS = ("U", "U1", "T", "RHS", "VEL_X", "VEL_Y", "RHO", "E", "P", "X", "Y", "W_X", "W_Y", "XPOS",
          "M", "AREA", "DNX", "HH", "DT", "SHOC", "T_SUGN3", "LAP_SPARSE", "LAP_DIAG")


@pytest.mark.parametrize("nr, nt, pe", [(24, 48, 0), (24, 48, 4), (40, 512, 0), (40, 513, 0),
                                        (260, 400, 0)])
@pytest.mark.parametrize("precision, renumber", [(0, 0), (1, 1), (2, 0)])
@pytest.mark.parametrize("gcl", [-1, 0, 1])
def test_steps_of_one_call(nr, nt, pe, precision, renumber, gcl):
    cs = ellipse_case(nr, nt, re=1000.0)
    kw = dict(motion=1, motion_amp=0.05, motion_omega=0.2, gcl=gcl, precision=precision,
              renumber=renumber, patch_elems=pe if precision < 2 else 0)
    print(f"{nr} x {nt}, patches {pe}, precision {precision}, gcl {gcl}", flush=True)
    one, many = Session(cs, **kw), Session(cs, **kw)
    for n in (1, 3, 2):
        for _ in range(n):
            one.step(1)
            one.scalars()
            one.get("P")
        many.step(n)
        a, b = one.scalars(), many.scalars()
        assert a == b and np.isfinite(list(a.values())).all()
    assert a["FX1"] != 0.0 and a["HMIN"] > 0.0
    for k in FIELDS:
        x, y = one.get(k), many.get(k)
        assert np.isfinite(x).all() and x.tobytes() == y.tobytes(), k
