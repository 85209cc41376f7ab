"""Sessions of few element patches take other launches than large ones: a
thread per element, a stage's halo nodes formed by the next stage, step control
inside ESTAB, the forces in one block.  The patch size moves a small mesh from
one rule to the other.

Binary32 elements: a node's contributions add exactly in FP64, so every patch
shape and thread count gives the same bits.  FP64: each step from the oracle's
state within the 1e-12 bar of the path (norm-relative per component)."""
import numpy as np
import pytest

from cfd_amd.mesh import cylinder_case, ellipse_case
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# patches of the 41 x 80 mesh (6,400 triangles): 13; 400 (nodes in more than
# four patches); 1,067 and 6,400 (halo kernel, step control of its own)
SHAPES = [(512, 0), (512, 64), (16, 0), (16, 256), (6, 0), (1, 0)]


def _run(cs, pe, block, **kw):
    from cfd_amd.solver import Session
    S = Session(cs, patch_elems=pe, patch_block=block, **kw)
    S.step(4)
    out = {k: S.get(k) for k in ("U", "T", "RHS", "VEL_X", "P", "DT", "SHOC", "X")}
    sc = S.scalars()
    out["scalars"] = np.array([sc[k] for k in ("DTMIN", "TIME", "ITER", "BANDERA", "DTMIN1", "FX1",
                                               "FY1", "RM1", "FVX1", "FVY1")])
    S.close()
    return out


@pytest.mark.parametrize("renumber", [0, 1])
@pytest.mark.parametrize("itlocal", [0, 7])
def test_patch_shapes_give_the_same_bits(renumber, itlocal):
    cs = cylinder_case(41, 80, mach=0.5, re=300.0, itlocal=itlocal)
    ref = _run(cs, *SHAPES[0], precision=1, renumber=renumber)
    assert np.isfinite(ref["U"]).all()
    for pe, block in SHAPES[1:]:
        print(f"patches of {pe} elements, block {block}", flush=True)
        got = _run(cs, pe, block, precision=1, renumber=renumber)
        for k in ref:
            assert np.array_equal(ref[k], got[k]), (pe, block, k)


@pytest.mark.parametrize("nt", [64, 65, 512, 513])   # 1, 2, 8 and 9 pieces of the forces
def test_forces_in_one_block_or_two(nt):
    from cfd_amd.api import MeshContext
    cs = cylinder_case(6, nt, mach=0.5, re=300.0)
    m = cs.mesh
    rng = np.random.default_rng(nt)
    g = orc_geometry(m)
    P, T = rng.uniform(1, 2, m.npoin), rng.uniform(200, 300, m.npoin)
    vx, vy = rng.standard_normal(m.npoin), rng.standard_normal(m.npoin)
    iset = cs.lists["iset"]
    mc = MeshContext(m.inpoel, m.npoin)
    fx, fy = mc.force_visc(iset, m.x, m.y, P, T, vx, vy, g["dNx"], g["dNy"], cs.t_inf)
    # the edges' terms one by one, summed as the kernels do: 64 edges by a tree
    # (lane l adds lane l + 32, 16, ...), the pieces in order by lane, a tree
    one = np.array([mc.force_visc(e[None, :], m.x, m.y, P, T, vx, vy, g["dNx"], g["dNy"], cs.t_inf)
                    for e in iset])

    def tree(v):
        v = np.concatenate([v, np.zeros(64 - v.size)])
        for off in (32, 16, 8, 4, 2, 1):
            v[:64 - off] = v[:64 - off] + v[off:]
        return v[0]
    for k, f in enumerate((fx, fy)):
        pieces = np.array([tree(one[b:b + 64, k]) for b in range(0, nt, 64)])
        assert f == tree(0.0 + pieces)


def orc_geometry(m):
    from cfd_amd.api import MeshContext
    return MeshContext(m.inpoel, m.npoin).deriv(m.x, m.y)


@pytest.mark.parametrize("moving", [False, True])
@pytest.mark.parametrize("pe, block", [(384, 0), (384, 192), (16, 0), (1, 0)])
def test_fp64_step_from_the_oracle(moving, pe, block):
    from cfd_amd.solver import Session
    cs = ellipse_case(25, 48, re=1000.0) if moving else cylinder_case(41, 80, mach=0.5, re=300.0)
    o = orc.OracleSolver(cs)
    for _ in range(3):
        o.step()
    S = Session(cs, patch_elems=pe, patch_block=block)
    S.set_state(o.state())
    if moving:
        S.set_scalars(DISN2=o.disn2)
    o.step()
    S.step(1)
    ref, got = o.state(), S.state()
    for name in ("U", "RHS"):
        for k in range(4):
            a, b = got[name][:, k], ref[name][:, k]
            assert np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(b), (name, k)
    assert got["DTMIN"] == ref["DTMIN"] and got["TIME"] == ref["TIME"]


@pytest.mark.parametrize("nr, nt, precision, viscous", [
    (9, 33, 0, True), (24, 64, 1, True), (20, 65, 0, False), (150, 512, 0, True),
    (150, 513, 1, True), (30, 96, 2, True),
])
def test_forces_of_many_steps_in_one_call(nr, nt, precision, viscous):
    """The steps of one call leave their forces to the next step's deltat (up to
    512 edges): after every number of steps they are those of steps called one
    by one, with and without FORCE_VISC, bit for bit."""
    from cfd_amd.solver import Session
    cs = cylinder_case(nr, nt)
    if not viscous:
        cs.fmu = cs.fk = 0.0
    print(f"forces on {nt} edges, precision {precision}", flush=True)
    one, many = Session(cs, precision=precision), Session(cs, precision=precision)
    names = ("FX1", "FY1", "RM1", "FVX1", "FVY1", "PCG_ITX", "PCG_ITY", "TIME")
    for n in (1, 2, 5, 1):
        for _ in range(n):
            one.step(1)
        many.step(n)
        a, b = one.scalars(), many.scalars()
        assert np.isfinite([a[k] for k in names]).all()
        assert [a[k] for k in names] == [b[k] for k in names]
    # (after the first step the pressure is uniform and its force closes to 0)
    assert a["FX1"] != 0.0 and (a["FVX1"] != 0.0) == viscous
