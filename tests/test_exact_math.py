"""The kernels' quotients and roots (cfd_amd/csrc/crmath.hpp: shared reciprocals,
no scaling steps) are the correctly rounded ones: cfd_deltat and the shock
parameter of cfd_estab bit for bit against numpy's '/' and sqrt in the same
order of operations, for velocities over many orders of magnitude and for the
special values (a gas at rest, zero gradients, infinite lengths).  The
temperature is T_inf everywhere, so that the power in both is 1**1.5 = 1."""
import numpy as np
import pytest

from cfd_amd.api import MeshContext, consts_of
from cfd_amd.mesh import cylinder_case

pytestmark = pytest.mark.gpu


def _state(cs, scale, rest, seed):
    rng = np.random.default_rng(seed)
    n = cs.npoin
    speed = 0.0 if rest else scale * np.hypot(cs.u_inf, cs.v_inf)
    U = np.ones((n, 4))
    if not rest:
        U[:, 0] = rng.uniform(0.5, 2.0, n)
    T = np.full(n, cs.t_inf)
    vx, vy = speed * rng.standard_normal(n), speed * rng.standard_normal(n)
    return U, T, vx, vy


@pytest.mark.parametrize("scale, rest", [(1.0, False), (1e-6, False), (1e6, False), (1e-30, False),
                                         (1.0, True)])
def test_deltat_and_shock_parameter_bitwise(scale, rest):
    cs = cylinder_case(13, 29, mach=0.5, re=200.0)
    m = cs.mesh
    mc = MeshContext(m.inpoel, m.npoin)
    k = consts_of(cs)
    g = mc.deriv(m.x, m.y)
    U, T, vx, vy = _state(cs, scale, rest, 3)
    z = np.zeros(cs.npoin)
    gm = np.full(cs.npoin, cs.gama)
    DT, dtmin = mc.deltat(k, g["area"], T, vx, vy, z, z)
    n = m.inpoel - 1
    hh = np.sqrt(2.0 * g["area"])
    vu, vv = np.abs(vx[n]).max(1), np.abs(vy[n]).max(1)
    vel = np.sqrt(vu * vu + vv * vv)
    t = (T[n[:, 0]] + T[n[:, 1]] + T[n[:, 2]]) / 3.0
    assert np.all(t == cs.t_inf)
    fmu = 0.017 * 1.0 * (cs.t_inf + 110.0) / (t + 110.0)
    pe = (vel * hh) / (2.0 * fmu)
    al = np.where(pe / 3.0 < 1.0, pe / 3.0, 1.0)
    du = 1.0 / (4.0 * fmu / (hh * hh) + al * vel / hh)
    dc = 1.0 / (4.0 * fmu / (hh * hh))
    ref = cs.fsafe / (1.0 / dc + 1.0 / du)
    assert dtmin == ref.min()
    assert np.array_equal(DT, np.minimum(ref, 10.0 * dtmin))
    sh, _, _, _ = mc.ESTAB(k, U, T, gm, vx, vy, z, z, g["dNx"], g["dNy"], dtmin)
    r = U[n, 0]
    drx = r[:, 0] * g["dNx"][:, 0] + r[:, 1] * g["dNx"][:, 1] + r[:, 2] * g["dNx"][:, 2]
    dry = r[:, 0] * g["dNy"][:, 0] + r[:, 1] * g["dNy"][:, 1] + r[:, 2] * g["dNy"][:, 2]
    dr2 = np.sqrt(drx * drx + dry * dry) + 1.0e-20
    rx, ry = drx / dr2, dry / dr2
    gme = (gm[n[:, 0]] + gm[n[:, 1]] + gm[n[:, 2]]) / 3.0
    cc = np.sqrt(gme * cs.fr * t)
    hj = np.zeros(cs.nelem)
    for i in range(3):
        hj = hj + np.abs(rx * g["dNx"][:, i] + ry * g["dNy"][:, i])
    with np.errstate(divide="ignore"):
        hj = 2.0 / hj
    hj = np.where(hj > 10.0, 0.0, hj)
    tr1 = dr2 * hj / ((r[:, 0] + r[:, 1] + r[:, 2]) / 3.0)
    ref = (tr1 + tr1 * tr1) * 0.5 * (cc * cc) * (hj / (2.0 * cc))
    assert np.array_equal(sh, ref)
