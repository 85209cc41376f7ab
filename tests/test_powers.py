"""x^(3/2) of the kernels (cfd_amd/csrc/crmath.hpp) where it lies exactly between two
doubles: x = k^2 with an odd k whose cube has 54 bits.  cfd_deltat at the
temperatures k^2 (T_inf = 1, no velocity, one element per k) bit for bit against
numpy in the same order of operations, the power from integer arithmetic, rounded
to even."""
import numpy as np
import pytest

from cfd_amd.api import MeshContext, consts_of
from cfd_amd.mesh import cylinder_case

pytestmark = pytest.mark.gpu


def test_three_halves_power_of_squares():
    k = np.array([k for k in range(208065, 262144, 2) if (k ** 3).bit_length() == 54])
    assert k.size > 20000
    n, ne = 3 * k.size, k.size
    mc = MeshContext(np.arange(1, n + 1, dtype=np.int32).reshape(ne, 3), n)
    c = consts_of(cylinder_case(13, 29, mach=0.5, re=200.0))
    c.t_inf = 1.0
    T = (k.astype(np.float64) ** 2).repeat(3)
    z, area = np.zeros(n), np.full(ne, 0.37)
    DT, dtmin = mc.deltat(c, area, T, z, z, z, z)
    t = T[::3]
    cube = np.array([float(int(q) ** 3) for q in k])
    hh = np.sqrt(2.0 * area)
    et = 0.017 * cube * (1.0 + 110.0) / (t + 110.0)
    visc = 4.0 * et / (hh * hh)
    du = 1.0 / (visc + (0.0 * hh) / (2.0 * et) / 3.0 * 0.0 / hh)
    ref = c.fsafe / (1.0 / (1.0 / visc) + 1.0 / du)
    assert dtmin == ref.min()
    off = int(np.sum(DT != ref))
    assert off == 0, f"{off} of {ne} elements"
