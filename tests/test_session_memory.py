"""What a session keeps on the device goes with what it does: the elements' weights
in the mesh-motion matrix (8 bytes a triangle) belong to moving meshes, whose every
step needs them; a fixed mesh forms its matrix once."""
import ctypes as C

import pytest

from cfd_amd._lib import lib
from cfd_amd.api import MeshContext
from cfd_amd.mesh import Case, acoustic_fsafe, ogrid
from cfd_amd.solver import Session

pytestmark = pytest.mark.gpu


def _free():
    lib()                                   # loads libcfd_amd.so and its runtime
    hip = C.CDLL("libamdhip64.so.7")        # the same, already loaded, instance
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_fixed_meshes_keep_no_matrix_weights():
    mesh = ogrid(1001, 1000, "circle")      # 2,000,000 triangles: 16 MB of weights
    ctx = MeshContext(mesh.inpoel, mesh.npoin)
    used = {0: [], 1: []}
    for _ in range(3):
        for moving in (0, 1):
            cs = Case(name="case", mesh=mesh, mach=0.5, re=500.0, moving=moving,
                      fsafe=acoustic_fsafe(0.5))
            before = _free()
            S = Session(cs, mesh=ctx)
            S.sync()
            used[moving].append(before - _free())
            S.close()
    print("fixed, moving: " + ", ".join(f"{a / 1e6:.1f} {b / 1e6:.1f}" for a, b in zip(*used.values())))
    # besides the weights a moving mesh has its matrix in the solves' order: seven
    # values, 16-bit columns and a length per node.  The first ones also pay for
    # code objects and pools.
    ell = (7 * (8 + 2) + 1) * mesh.npoin
    assert min(used[1][1:]) - max(used[0][1:]) >= ell + 8 * mesh.nelem - (4 << 20)
