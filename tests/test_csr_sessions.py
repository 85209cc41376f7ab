"""Moving-mesh sessions whose matrix has no ELL copy (a row longer than 16 entries):
both mesh solves from the CSR rows.  The mesh is the pitching ellipse's with a star
of 17 triangles beside it, its rim held and its hub free: the hub's row is the long
one, and contributes nothing but zeros to every sum, so the ellipse's coordinates
are bit for bit those of the ellipse alone, whose solves read the copy (and run in
one launch where they are small)."""
import copy

import numpy as np
import pytest

from cfd_amd.mesh import Mesh, ellipse_case
from cfd_amd.solver import Session

pytestmark = pytest.mark.gpu

RIM = 17


def _with_star(cs):
    m, n = cs.mesh, cs.npoin
    ang = 2 * np.pi * np.arange(RIM) / RIM
    x = np.concatenate([m.x, [200.0], 200.0 + 60.0 * np.cos(ang)])
    y = np.concatenate([m.y, [0.0], 60.0 * np.sin(ang)])
    rim = n + 2 + np.arange(RIM)
    tri = np.stack([np.full(RIM, n + 1), rim, np.roll(rim, -1)], axis=1).astype(np.int32)
    new = copy.copy(cs)
    new.mesh = Mesh(x, y, np.concatenate([m.inpoel, tri]), m.nr, m.nt, m.body)
    new.lists = dict(cs.lists)
    new.lists["ilaux"] = np.concatenate([cs.lists["ilaux"], rim]).astype(np.int32)
    new.lists["nfix_move"] = int(cs.lists["nfix_move"]) + RIM
    return new


@pytest.mark.parametrize("nr, nt", [(24, 48), (60, 100), (420, 401), (660, 401)])
@pytest.mark.parametrize("warm, rel", [(0, 1), (2, 1), (2, 0)])
def test_solves_from_csr_rows(nr, nt, warm, rel):
    cs = ellipse_case(nr, nt)
    out = []
    for case in (cs, _with_star(cs)):
        S = Session(case, motion=1, motion_amp=0.05, motion_omega=0.2, pcg_rel=rel,
                    pcg_tol=1e-6 if rel else 0.0, pcg_maxit=20000 if rel else 0, warm_start=warm)
        print(f"mesh solves on {case.npoin} nodes, warm start {warm}, rel {rel}", flush=True)
        S.step(2 if nr > 400 else 6)
        sc = S.scalars()
        out.append([S.get(k)[:cs.npoin].tobytes() for k in ("X", "Y", "XPOS", "YPOS", "W_X")]
                   + [sc["PCG_ITSUM"], sc["PCG_UNCONV"], sc["WS_SOLVES"], sc["WS_LEARNED"]])
    assert out[0] == out[1]
    assert out[0][6] == 0 and (not rel or out[0][5] > 10)
