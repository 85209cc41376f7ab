"""Fields of renumbered sessions and of batches on both sides of the size from which a
kernel, and not the host, puts them into the caller's order: what is written is
read back, reaches the same entities as in a session in the caller's numbering (a
step on a fixed mesh from them gives the same bits), and a batch's cases read like
their sessions."""
import numpy as np
import pytest

from cfd_amd.batch import Batch
from cfd_amd.mesh import cylinder_case
from cfd_amd.solver import Session

pytestmark = pytest.mark.gpu

NODE = ("U", "U1", "T", "VEL_X", "VEL_Y", "RHO", "E", "P", "M", "GAMM", "X")
ELEM = ("DT", "SHOC", "T_SUGN1", "AREA", "DNX", "HH")


# U of 40,000 doubles on the host, the next size by the kernel; the elements' fields
# and nodes' scalars change over at other sizes
@pytest.mark.parametrize("nr, nt", [(5, 12), (100, 100), (101, 100), (70, 96), (200, 200),
                                    (200, 201), (130, 160)])
def test_written_fields_arrive(nr, nt):
    cs = cylinder_case(nr, nt, mach=0.5, re=300.0)
    rng = np.random.default_rng(nr)
    a, b = Session(cs, precision=1), Session(cs, precision=1, renumber=1)
    print(f"{cs.npoin} nodes, {cs.nelem} triangles", flush=True)
    for k in ("LAP_SPARSE", "DNY", "RHS"):
        v = rng.standard_normal(b.get(k).shape)
        b.set(k, v)
        assert np.array_equal(b.get(k), v), k
    b.set("DNY", a.get("DNY"))
    a.step(3)
    for k in ("U", "U1", "T", "VEL_X", "VEL_Y", "RHO", "E", "P"):
        v = a.get(k)
        a.set(k, v)
        b.set(k, v)
    sc = a.scalars()
    b.set_scalars(**{k: sc[k] for k in ("TIME", "ITER", "DTMIN", "DTMIN1", "BANDERA")})
    a.step(1)
    b.step(1)
    for k in NODE + ELEM:
        assert np.array_equal(a.get(k), b.get(k)), k


def test_cases_of_a_batch_read_like_their_sessions():
    cases = [cylinder_case(nr, nt, mach=0.5, re=300.0) for nr, nt in ((20, 31), (100, 100), (101, 101))]
    B = Batch(cases, precision=1)
    B.step(2)
    for k, cs in enumerate(cases):
        S = Session(cs, precision=1)
        S.step(2)
        for f in NODE + ELEM:
            assert np.array_equal(B.get(k, f), S.get(f)), (k, f)
