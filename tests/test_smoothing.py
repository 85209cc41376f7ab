"""Start-up mesh smoothing: smoothing_mod::smoothing (smoothing.f90:21-75).

The reference's smoothing.f90 does not compile with flang (smoothing.f90:45
compares LOGICALs with ==), so the oracle's restatement (orc_smoothing,
reference node order) is pinned here by what the mathematics fixes:

- a regular hexagon with its centre displaced: the Laplacian pass puts the
  centre at the rim's mean (the origin), every element becomes equilateral
  and the sweeps stop after the first;
- a mesh with no element below the quality bound is returned untouched;
- one free node in a random star (rim fixed): the Laplacian passes can only
  put it at the rim's mean or leave it, so after them its worst element is
  the better of the two; the sweeps then never make it worse, never beat the
  brute-force max-min optimum over a fine grid of positions (by more than the
  grid's resolution), and close at least a fifth of the remaining gap to it
  (a sign or index slip in the gradient, the step or the tries leaves the
  node where the Laplacian put it);
- the sweeps one at a time (the oracle stopped after 1, 2, ... sweeps): the
  worst element around the free node never gets worse from one sweep to the
  next (the acceptance rule);
- tol_move mode: each Laplacian step has L1 length 1.5 tol_move and each
  optimisation step at most tol_move / 100, so no node moves further than
  7 tol_move in L1; on the displaced hexagon both Laplacian steps are taken
  straight towards the centre, so the centre moves 3 tol_move (L1) there,
  give or take the one sweep's 0.04 tol_move;
- on jittered O-grids: fixed nodes stay put bit for bit, the worst element
  only improves, no element inverts.

GPU (cfd_smoothing): order 0 (the reference's node order) equals the oracle
bit for bit on whole meshes, with and without tol_move and on a second call
of one context (the tol_move mode stays on, as the reference's module state
does); order 1 (colour by colour) equals it bit for bit where the order
cannot matter (free nodes that share no element), and on whole meshes keeps
the same invariants and reaches a comparable worst element.
"""
import numpy as np
import pytest

from cfd_amd.mesh import cylinder_case, ellipse_case
from oracle import oracle as orc

TWOSQRT3 = 3.46410161513775


def quality(inpoel, X, Y):
    a = np.asarray(inpoel) - 1
    X1, X2, X3 = X[a[:, 0]], X[a[:, 1]], X[a[:, 2]]
    Y1, Y2, Y3 = Y[a[:, 0]], Y[a[:, 1]], Y[a[:, 2]]
    ar = X2 * Y3 + X3 * Y1 + X1 * Y2 - (X2 * Y1 + X3 * Y2 + X1 * Y3)
    l = ((X3 - X2) ** 2 + (Y3 - Y2) ** 2) + ((X1 - X3) ** 2 + (Y1 - Y3) ** 2) + \
        ((X2 - X1) ** 2 + (Y2 - Y1) ** 2)
    return TWOSQRT3 * ar / l


def hexagon(cx=0.5, cy=0.2):
    ang = np.arange(6) * np.pi / 3
    X = np.concatenate([[cx], np.cos(ang)])
    Y = np.concatenate([[cy], np.sin(ang)])
    inp = np.array([[1, 2 + i, 2 + (i + 1) % 6] for i in range(6)], np.int32)
    fixed = np.ones(7, np.int32)
    fixed[0] = 0
    return inp, X, Y, fixed


def star(rng, k):
    ang = np.linspace(0, 2 * np.pi, k, endpoint=False) + rng.uniform(-0.3, 0.3, k)
    r = rng.uniform(0.6, 1.4, k)
    X = np.concatenate([[0.25 * rng.standard_normal()], r * np.cos(ang)])
    Y = np.concatenate([[0.25 * rng.standard_normal()], r * np.sin(ang)])
    inp = np.array([[1, 2 + i, 2 + (i + 1) % k] for i in range(k)], np.int32)
    fixed = np.ones(k + 1, np.int32)
    fixed[0] = 0
    return inp, X, Y, fixed


def brute_maxmin(inp, X, Y, n=401):
    g = np.linspace(-1.0, 1.0, n)
    gx, gy = np.meshgrid(g, g)
    a = inp - 1
    best = -np.inf
    for q in range(inp.shape[0]):  # min over the star's elements on the whole grid
        XX = [np.full_like(gx, X[j]) if j else gx for j in a[q]]
        YY = [np.full_like(gy, Y[j]) if j else gy for j in a[q]]
        X1, X2, X3 = XX
        Y1, Y2, Y3 = YY
        ar = X2 * Y3 + X3 * Y1 + X1 * Y2 - (X2 * Y1 + X3 * Y2 + X1 * Y3)
        l = ((X3 - X2) ** 2 + (Y3 - Y2) ** 2) + ((X1 - X3) ** 2 + (Y1 - Y3) ** 2) + \
            ((X2 - X1) ** 2 + (Y2 - Y1) ** 2)
        m = TWOSQRT3 * ar / l
        best = m if q == 0 else np.minimum(best, m)
    return float(best.max())


def ogrid_case(which):
    cs = cylinder_case(16, 32) if which == "cyl" else ellipse_case(24, 48)
    fixed = np.zeros(cs.npoin, np.int32)
    for k in ("i_m", "ifm"):  # SMOOTH_FIX = moving + fixed-move lists (ns2DComp.ALE.f90:62-74)
        fixed[np.asarray(cs.lists[k], int) - 1] = 1
    return cs, fixed


# ---------------------------------------------------------------------------
# oracle pinning (CPU)
# ---------------------------------------------------------------------------
def test_oracle_hexagon_closed_form():
    inp, X, Y, fixed = hexagon()
    assert quality(inp, X, Y).min() < 0.85
    Xs, Ys, sweeps, h = orc.smoothing(inp, 7, X, Y, fixed)
    assert abs(Xs[0]) < 1e-15 and abs(Ys[0]) < 1e-15
    assert np.array_equal(Xs[1:], X[1:]) and np.array_equal(Ys[1:], Y[1:])
    assert np.all(np.abs(quality(inp, Xs, Ys) - TWOSQRT3 / (2 * np.sqrt(3))) < 1e-14)
    assert sweeps == 1
    # H_MIN_GLOBAL = min(1, |area| / L1 perimeter) over the initial elements
    a = inp - 1
    ar = np.abs(X[a[:, 1]] * Y[a[:, 2]] + X[a[:, 2]] * Y[a[:, 0]] + X[a[:, 0]] * Y[a[:, 1]]
                - (X[a[:, 1]] * Y[a[:, 0]] + X[a[:, 2]] * Y[a[:, 1]] + X[a[:, 0]] * Y[a[:, 2]]))
    per = sum(np.abs(X[a[:, i]] - X[a[:, j]]) + np.abs(Y[a[:, i]] - Y[a[:, j]])
              for i, j in ((2, 1), (0, 2), (1, 0)))
    assert h == pytest.approx(min(1.0, float((ar / per).min())), rel=1e-14)


def test_oracle_good_mesh_untouched():
    inp, X, Y, fixed = hexagon(0.0, 0.0)
    assert quality(inp, X, Y).min() > 0.85
    Xs, Ys, sweeps, _ = orc.smoothing(inp, 7, X, Y, fixed)
    assert sweeps == 0 and np.array_equal(Xs, X) and np.array_equal(Ys, Y)


def test_oracle_single_node_climbs_towards_the_maxmin_optimum():
    rng = np.random.default_rng(1)
    checked = 0
    for _ in range(40):
        k = int(rng.integers(4, 9))
        inp, X, Y, fixed = star(rng, k)
        q0 = quality(inp, X, Y).min()
        if q0 >= 0.85:  # nothing smoothable: returned as is
            continue
        best = brute_maxmin(inp, X, Y)
        Xc, Yc = X.copy(), Y.copy()
        Xc[0], Yc[0] = X[1:].mean(), Y[1:].mean()
        q_lap = max(q0, quality(inp, Xc, Yc).min())
        Xs, Ys, sweeps, _ = orc.smoothing(inp, k + 1, X, Y, fixed)
        q1 = quality(inp, Xs, Ys).min()
        assert q_lap - 1e-12 <= q1 <= best + 0.005, (k, q0, q_lap, q1, best)
        if q_lap < 0.85 and best - q_lap > 0.005:
            assert q1 >= q_lap + 0.2 * (best - q_lap), (k, q0, q_lap, q1, best)
            checked += 1
    assert checked >= 20


def test_oracle_sweeps_never_worsen_the_node():
    rng = np.random.default_rng(2)
    checked = 0
    for _ in range(30):
        k = int(rng.integers(4, 9))
        inp, X, Y, fixed = star(rng, k)
        if quality(inp, X, Y).min() >= 0.85:
            continue
        prev = -np.inf
        for ms in range(0, 6):
            Xs, Ys, _, _ = orc.smoothing(inp, k + 1, X, Y, fixed, max_sweeps=ms)
            q = quality(inp, Xs, Ys).min()
            assert q >= prev - 1e-15, (k, ms, q, prev)
            prev = q
        checked += 1
    assert checked >= 15


def test_oracle_tol_move_laplacian_step_on_the_hexagon():
    inp, X, Y, fixed = hexagon()
    tm = np.full(7, 0.05)
    Xs, Ys, sweeps, _ = orc.smoothing(inp, 7, X, Y, fixed, tol_move=tm)
    l1 = abs(Xs[0] - X[0]) + abs(Ys[0] - Y[0])
    assert abs(l1 - 3 * 0.05) <= 0.04 * 0.05, l1
    # straight towards the centre
    assert abs(Xs[0] * Y[0] - Ys[0] * X[0]) < 0.04 * 0.05
    assert sweeps == 1


def test_oracle_tol_move_bounds_the_moves():
    for which in ("cyl", "ell"):
        cs, fixed = ogrid_case(which)
        m = cs.mesh
        rng = np.random.default_rng(3)
        dX = 1e-3 * rng.standard_normal(cs.npoin)
        dY = 1e-3 * rng.standard_normal(cs.npoin)
        tm = np.abs(dX) + np.abs(dY)
        Xs, Ys, sweeps, _ = orc.smoothing(m.inpoel, cs.npoin, m.x, m.y, fixed, tol_move=tm)
        l1 = np.abs(Xs - m.x) + np.abs(Ys - m.y)
        assert sweeps >= 1 and np.count_nonzero(l1) > 0
        assert np.all(l1 <= 7 * tm * (1 + 1e-12))
        assert quality(m.inpoel, Xs, Ys).min() >= quality(m.inpoel, m.x, m.y).min()


@pytest.mark.parametrize("which", ["cyl", "ell"])
def test_oracle_ogrid_invariants(which):
    cs, fixed = ogrid_case(which)
    m = cs.mesh
    q0 = quality(m.inpoel, m.x, m.y)
    Xs, Ys, sweeps, _ = orc.smoothing(m.inpoel, cs.npoin, m.x, m.y, fixed)
    q1 = quality(m.inpoel, Xs, Ys)
    f = fixed == 1
    assert np.array_equal(Xs[f], m.x[f]) and np.array_equal(Ys[f], m.y[f])
    assert 1 <= sweeps <= 100
    assert q1.min() > q0.min() and q1.min() > 0


# ---------------------------------------------------------------------------
# device (cfd_smoothing)
# ---------------------------------------------------------------------------
def _ctx(inp, npoin):
    from cfd_amd.api import MeshContext
    return MeshContext(inp, npoin)


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["hex", "cyl", "ell"])
def test_reference_order_bitwise(which):
    if which == "hex":
        inp, X, Y, fixed = hexagon()
        n = 7
    else:
        cs, fixed = ogrid_case(which)
        inp, X, Y, n = cs.mesh.inpoel, cs.mesh.x, cs.mesh.y, cs.npoin
    mc = _ctx(inp, n)
    Xg, Yg, sg, hg = mc.smoothing(X, Y, fixed, order=0)
    Xo, Yo, so, ho = orc.smoothing(inp, n, X, Y, fixed)
    print(which, "sweeps", sg, so)
    assert (sg, hg) == (so, ho)
    assert np.array_equal(Xg, Xo) and np.array_equal(Yg, Yo)
    mc.close()


@pytest.mark.gpu
def test_reference_order_tol_move_and_its_module_state():
    cs, fixed = ogrid_case("cyl")
    m = cs.mesh
    rng = np.random.default_rng(5)
    dX = 1e-3 * rng.standard_normal(cs.npoin)
    dY = 1e-3 * rng.standard_normal(cs.npoin)
    tm = np.abs(dX) + np.abs(dY)
    mc = _ctx(m.inpoel, cs.npoin)
    Xg, Yg, sg, _ = mc.smoothing(m.x, m.y, fixed, dX, dY, order=0)
    Xo, Yo, so, _ = orc.smoothing(m.inpoel, cs.npoin, m.x, m.y, fixed, tol_move=tm)
    assert sg == so and np.array_equal(Xg, Xo) and np.array_equal(Yg, Yo)
    # a second call without dX, dY keeps the tol_move mode
    Xg2, Yg2, sg2, _ = mc.smoothing(Xg, Yg, fixed, order=0)
    Xo2, Yo2, so2, _ = orc.smoothing(m.inpoel, cs.npoin, Xo, Yo, fixed, tol_move=tm)
    assert sg2 == so2 and np.array_equal(Xg2, Xo2) and np.array_equal(Yg2, Yo2)
    mc.close()


@pytest.mark.gpu
def test_colour_order_equals_the_reference_where_order_cannot_matter():
    rng = np.random.default_rng(7)
    for _ in range(10):
        k = int(rng.integers(4, 9))
        inp, X, Y, fixed = star(rng, k)
        mc = _ctx(inp, k + 1)
        Xg, Yg, sg, _ = mc.smoothing(X, Y, fixed, order=1)
        Xo, Yo, so, _ = orc.smoothing(inp, k + 1, X, Y, fixed)
        assert sg == so and np.array_equal(Xg, Xo) and np.array_equal(Yg, Yo)
        mc.close()
    # an O-grid whose free nodes share no element (every other node of every
    # other interior ring, the rest fixed)
    cs, fixed = ogrid_case("ell")
    m = cs.mesh
    fx = np.ones(cs.npoin, np.int32)
    for r in range(2, m.nr - 2, 2):
        fx[m.node(r, np.arange(0, m.nt, 2)) - 1] = 0
    mc = _ctx(m.inpoel, cs.npoin)
    Xg, Yg, sg, _ = mc.smoothing(m.x, m.y, fx, order=1)
    Xo, Yo, so, _ = orc.smoothing(m.inpoel, cs.npoin, m.x, m.y, fx)
    assert sg == so and np.array_equal(Xg, Xo) and np.array_equal(Yg, Yo)
    assert np.count_nonzero(Xg != m.x) > 10
    mc.close()


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["cyl", "ell"])
def test_colour_order_whole_mesh(which):
    cs, fixed = ogrid_case(which)
    m = cs.mesh
    mc = _ctx(m.inpoel, cs.npoin)
    Xg, Yg, sg, _ = mc.smoothing(m.x, m.y, fixed, order=1)
    Xo, Yo, so, _ = orc.smoothing(m.inpoel, cs.npoin, m.x, m.y, fixed)
    q0, qg, qo = (quality(m.inpoel, a, b) for a, b in ((m.x, m.y), (Xg, Yg), (Xo, Yo)))
    print(which, "worst element: start %.4f, reference order %.4f (%d sweeps), by colour %.4f "
          "(%d sweeps)" % (q0.min(), qo.min(), so, qg.min(), sg))
    f = fixed == 1
    assert np.array_equal(Xg[f], m.x[f]) and np.array_equal(Yg[f], m.y[f])
    assert qg.min() > q0.min() and qg.min() > 0
    assert qg.min() >= 0.8 * qo.min()
    # deterministic
    Xg2, Yg2, _, _ = mc.smoothing(m.x, m.y, fixed, order=1)
    assert np.array_equal(Xg, Xg2) and np.array_equal(Yg, Yg2)
    mc.close()


@pytest.mark.gpu
def test_colour_order_at_the_bench_size():
    """Order 1 on the cylinder O-grid 1024 x 2048 (2,097,152 nodes): fixed
    nodes held, the worst element improved, no element inverted, and the
    wall time printed (order 0 is refused at this size)."""
    import time
    from cfd_amd._lib import CfdError
    cs = cylinder_case(1024, 2048)
    m = cs.mesh
    fixed = np.zeros(cs.npoin, np.int32)
    for k in ("i_m", "ifm"):
        fixed[np.asarray(cs.lists[k], int) - 1] = 1
    mc = _ctx(m.inpoel, cs.npoin)
    with pytest.raises(CfdError, match="65536"):
        mc.smoothing(m.x, m.y, fixed, order=0)
    t0 = time.perf_counter()
    Xg, Yg, sg, _ = mc.smoothing(m.x, m.y, fixed, order=1)
    sec = time.perf_counter() - t0
    q0, qg = quality(m.inpoel, m.x, m.y), quality(m.inpoel, Xg, Yg)
    print(f"order 1 at 2,097,152 nodes: {sec:.2f} s, {sg} sweeps, worst element "
          f"{q0.min():.4f} -> {qg.min():.4f}, mean {q0.mean():.4f} -> {qg.mean():.4f}")
    f = fixed == 1
    assert np.array_equal(Xg[f], m.x[f]) and np.array_equal(Yg[f], m.y[f])
    assert qg.min() > q0.min() and qg.min() > 0
    mc.close()


@pytest.mark.gpu
def test_smoothing_refusals():
    from cfd_amd._lib import CfdError
    # 21 elements around one node (the reference's MAX_ELEM_PER_NODE is 20)
    k = 21
    ang = np.linspace(0, 2 * np.pi, k, endpoint=False)
    X = np.concatenate([[0.1], np.cos(ang)])
    Y = np.concatenate([[0.0], np.sin(ang)])
    inp = np.array([[1, 2 + i, 2 + (i + 1) % k] for i in range(k)], np.int32)
    fixed = np.ones(k + 1, np.int32)
    fixed[0] = 0
    mc = _ctx(inp, k + 1)
    with pytest.raises(CfdError, match="20 elements"):
        mc.smoothing(X, Y, fixed, order=1)
    with pytest.raises(CfdError, match="order"):
        mc.smoothing(X, Y, fixed, order=2)
    with pytest.raises(CfdError, match="together"):
        mc.smoothing(X, Y, fixed, dX=np.zeros(k + 1), order=1)
    mc.close()


def _renumbered(m, seed):
    """The mesh with its nodes in random order: neighbours far apart."""
    p = np.random.default_rng(seed).permutation(m.npoin)
    X, Y = np.empty(m.npoin), np.empty(m.npoin)
    X[p], Y[p] = m.x, m.y
    return (p[m.inpoel - 1] + 1).astype(np.int32), X, Y, p


@pytest.mark.gpu
@pytest.mark.parametrize("nr, nt, shuffle", [
    (3, 5, False), (9, 64, False), (33, 65, False), (24, 40, True), (70, 130, False),
    (98, 98, False),        # 9,604 nodes: about the most whose positions fit LDS
    (90, 120, False),       # 10,800 nodes: positions in global memory
])
def test_reference_order_waves_bitwise(nr, nt, shuffle):
    """Order 0's passes run side by side, a block each: the chunks' edges, both
    places of the positions, and a numbering in which every node waits for far
    ones, bit for bit against the sequential oracle, with the sweep count."""
    from cfd_amd.api import MeshContext
    m = cylinder_case(nr, nt).mesh
    inp, X, Y = m.inpoel, m.x, m.y
    fixed = np.zeros(m.npoin, np.int32)
    fixed[: m.nt] = fixed[-m.nt:] = 1
    if shuffle:
        inp, X, Y, p = _renumbered(m, nr)
        f = np.zeros_like(fixed)
        f[p] = fixed
        fixed = f
    print(f"order 0 on {m.npoin} nodes", flush=True)
    xo, yo, n, h = orc.smoothing(inp, X.size, X, Y, fixed)
    xg, yg, ng, hg = MeshContext(inp, m.npoin).smoothing(X, Y, fixed)
    assert (n, h) == (ng, hg)
    assert np.array_equal(xo.view(np.int64), xg.view(np.int64))
    assert np.array_equal(yo.view(np.int64), yg.view(np.int64))


@pytest.mark.gpu
@pytest.mark.parametrize("k", [3, 8, 9, 16, 17, 20])
def test_reference_order_ring_sizes_bitwise(k):
    """One free node with k elements: every group width and its edges."""
    from cfd_amd.api import MeshContext
    for seed in range(4):
        inp, X, Y, fixed = star(np.random.default_rng(100 * k + seed), k)
        xo, yo, n, h = orc.smoothing(inp, X.size, X, Y, fixed)
        xg, yg, ng, hg = MeshContext(inp, X.size).smoothing(X, Y, fixed)
        assert (n, h) == (ng, hg)
        assert np.array_equal(xo, xg) and np.array_equal(yo, yg)
