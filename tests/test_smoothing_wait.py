"""Order 0's passes wait for each other on the GPU; a wait without progress ends.
With a limit far below what the first pass takes for its first nodes (64 updates
of about 3 us) the second one gives up: the call fails, the coordinates stay, and
the same context smooths bit for bit like the oracle once the limit is back."""
import ctypes as C

import numpy as np
import pytest

from cfd_amd._lib import CfdError, check, dptr, iptr, lib
from cfd_amd.api import MeshContext
from cfd_amd.mesh import cylinder_case
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr, nt", [(33, 65), (90, 120)])   # positions in LDS, in memory
def test_a_wait_without_progress_ends(nr, nt):
    m = cylinder_case(nr, nt).mesh
    fixed = np.zeros(m.npoin, np.int32)
    fixed[: m.nt] = fixed[-m.nt:] = 1
    mc = MeshContext(m.inpoel, m.npoin)
    x, y = m.x.copy(), m.y.copy()
    mc.set_smoothing_wait(1e-8)
    print(f"order 0 with a limit of 10 ns on {m.npoin} nodes", flush=True)
    with pytest.raises(CfdError, match="no progress"):
        check(lib().cfd_smoothing(mc.handle, dptr(x), dptr(y), iptr(fixed), None, None, 0,
                                  C.byref(C.c_int()), C.byref(C.c_double())))
    assert np.array_equal(x, m.x) and np.array_equal(y, m.y)
    mc.set_smoothing_wait(10.0)
    xg, yg, n, h = mc.smoothing(m.x, m.y, fixed)
    xo, yo, no, ho = orc.smoothing(m.inpoel, m.npoin, m.x, m.y, fixed)
    assert (n, h) == (no, ho) and np.array_equal(xg, xo) and np.array_equal(yg, yo)


def test_limits_out_of_range():
    mc = MeshContext(np.array([[1, 2, 3]], np.int32), 3)
    for s in (0.0, -1.0, 4000.0, float("nan")):
        with pytest.raises(CfdError, match="seconds"):
            mc.set_smoothing_wait(s)
