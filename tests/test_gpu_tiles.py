"""First-order Euler stages on tiles (tile.hip) where their face lists have
edges: fewer cells than a tile, exactly one tile, masked domains of one tile
and one cell more, remainders, grids of several levels whose interface tiles
overflow the halo and extra-face places, boundary conditions with and without
ghosts, and periodic images; each against the oracle."""
import numpy as np
import pytest

import oracle as O
from tests.scenarios import rel_l2

pytestmark = pytest.mark.gpu

TI = {"euler_forward": O.TI_EULER_FWD, "runge_kutta_2": O.TI_HEUN_RK2, "ssp_rk3": O.TI_SSP_RK3}
QUAD = [0.45, 0.55, 0.1, 0.2, 1.0, 1.0, -0.3, 0.1, 0.5, 0.4, 0.0, 0.0, 2.0, 1.5, 0.2, -0.2, 0.8, 0.9]
BALL = [0.5, 0.5, 0.5, 0.3, 0.1, -0.2, 0.0, 1.0, 10.0, 0.0, 0.0, 0.1, 0.125, 0.1]


def pair(nd, base, extra, radius, band, ti, bc, precision, kernel="tile"):
    import hom3_amd as H
    centre = [0.5, 0.4, 0.6][:nd]
    ic = (O.IC_FOUR_QUADRANT, QUAD) if nd == 2 else (O.IC_SPHERE, BALL)
    fixed = [0.1] * nd + [1.0, 2.5]
    if bc == "dirichlet":
        # the ghosts reflect the state at the fixed surface values, which only
        # stays physical for states near them
        ic = (O.IC_CONSTANT_PV, [0.1] * nd + [1.0, 0.4 * (2.5 - 0.5 * nd * 0.01)])
    cond = {"neumann": (O.BC_EULER_NEUMANN, lambda: H.euler.bc.Neumann()),
            "dirichlet": (O.BC_EULER_DIRICHLET, lambda: H.euler.bc.Dirichlet(fixed)),
            "periodic": (O.BC_PERIODIC, lambda: H.Periodic())}[bc]
    og = O.Grid(nd, [0.0] * nd, [1.0] * nd).min_level(base)
    g = H.Grid(nd, [0.0] * nd, [1.0] * nd, base)
    if extra:
        for r in radius if isinstance(radius, tuple) else (radius,):
            og.refine_region(base + extra, O.geom(O.GEOM_SPHERE, centre, [r]), band)
            g.refine_region(base + extra, H.Sphere(centre, r), band)
        og.balance()
        g.balance()
    o = O.Solver(og, O.phys(physics=O.PHYS_EULER, nd=nd, ti=TI[ti], cfl=0.2))
    prm = fixed if bc == "dirichlet" else []
    for i, geo in enumerate(O.cube_boundaries(nd, [0.0] * nd, [1.0] * nd)):
        o.append_bc(geo, cond[0], prm)
    o.set_ic(*ic)
    o.set_perturbation(5, 0.02)
    o.initialize()
    s = H.Solver(g, physics="euler", time_integration=ti, CFL=0.2, kernel=kernel, precision=precision)
    H.append_bcs(s, cond[1]())
    s.set_initial_condition(*ic)
    s.set_perturbation(5, 0.02)
    s.initialize()
    return o, s


# thin rings of finer cells: tiles of the coarse cells between them
RINGS = (2, 6, 1, tuple(0.02 + k * 3 / 64 for k in range(10)), 0.002)
# (nd, base, extra, radius, band): 16 and 64 cells; one tile; ragged tiles of
# refined grids; a ball refined twice and rings, whose tiles over the level
# interfaces have more halo cells and extra faces than places of their own
GRIDS = [(2, 2, 0, 0, 0), (3, 2, 0, 0, 0), (2, 4, 0, 0, 0), (2, 4, 2, 0.2, 0.05), (3, 3, 1, 0.25, 0.1),
         (3, 4, 2, 0.25, 0.02), RINGS]
PLACES = {2: (256, 256), 3: (384, 128)}  # halo cells and extra faces of a direction (tile.hpp)


def list_lengths(s, nd):
    """(halo cells, extra faces of each direction) of every tile of a solver
    with zero-gradient boundaries."""
    n, K = s.first_gc, 1 << (nd - 1)
    nb, fine = s.topology()["neighbors"], s.fine_faces()
    out = []
    for base in range(0, n, 256):
        end = min(n, base + 256)

        def away(x):
            return not base <= x < end
        halo, ext = 0, [0] * nd
        for c in range(base, end):
            for d in range(nd):
                lo, up = (c if v >= n else v for v in (int(nb[2 * d, c]), int(nb[2 * d + 1, c])))
                if lo >= 0:
                    halo += away(lo)
                else:
                    ext[d] += K
                    halo += sum(away(x) for x in fine[-lo - 2])
                if up < 0:
                    ext[d] += K
                    halo += sum(away(x) for x in fine[-up - 2])
                elif away(up) or up == c or int(nb[2 * d, up]) != c:  # not the lower face of a cell of the tile
                    ext[d] += 1
                    halo += away(up)
        out.append([halo] + ext)
    return np.array(out)


@pytest.mark.parametrize("grid", [(3, 4, 2, 0.25, 0.02), RINGS])
def test_grids_overflow_the_places(grid):
    """The grids above reach the lists past the places: halo cells read from
    memory, and extra faces in more than one chunk in every direction."""
    nd = grid[0]
    _, s = pair(*grid, "ssp_rk3", "neumann", "fp64")
    r = list_lengths(s, nd)
    nhc, ce = PLACES[nd]
    assert r[:, 0].max() > nhc
    for d in range(nd):
        assert r[:, 1 + d].max() > ce, d
    # and tiles that do not
    assert ((r[:, 0] <= nhc) & (r[:, 1:].max(1) <= ce)).any()


def _box(nd, level, shape, mask, ti):
    """A box of cells of a uniform grid, by its mask or its geometry: fixed
    values at its upper x side, zero gradients elsewhere."""
    import hom3_amd as H
    h = 1.0 / (1 << level)
    corner = [0.0] * nd if mask else [3 * h] * nd
    size = [k * h for k in shape]
    centre = [c + 0.5 * s for c, s in zip(corner, size)]
    fixed = [0.1] * nd + [1.0, 2.5]
    ic = [0.1] * nd + [1.0, 0.4 * (2.5 - 0.5 * nd * 0.01)]
    og = O.Grid(nd, [0.0] * nd, [1.0] * nd).min_level(level)
    g = H.Grid(nd, [0.0] * nd, [1.0] * nd, level)
    o = O.Solver(og, O.phys(physics=O.PHYS_EULER, nd=nd, ti=TI[ti], cfl=0.2))
    s = H.Solver(g, physics="euler", time_integration=ti, CFL=0.2, kernel="tile")
    for d in range(nd):
        for side in (0, 1):
            x = list(centre)
            x[d] = corner[d] + side * size[d]
            normal = [0.0] * nd
            normal[d] = -1.0 if side else 1.0
            dirichlet = d == 0 and side == 1
            o.append_bc(O.geom(O.GEOM_EDGE, x, normal), O.BC_EULER_DIRICHLET if dirichlet else O.BC_EULER_NEUMANN,
                        fixed if dirichlet else [])
            s.append_bc(H.Edge(x, normal), H.euler.bc.Dirichlet(fixed) if dirichlet else H.euler.bc.Neumann())
    if mask:
        # leaves in Morton order
        m = np.arange(1 << (nd * level))
        inside = np.ones(m.size, bool)
        for d in range(nd):
            inside &= sum(((m >> (nd * b + d)) & 1) << b for b in range(level)) < shape[d]
        o.set_domain_mask(inside)
        s.set_initial_domain(mask=inside)
    else:
        o.set_domain(O.geom(O.GEOM_SQUARE, centre, size, invert=True), +1)
        s.set_initial_domain(H.invert(H.Square(centre, size)), +1)
    for x in (o, s):
        x.set_ic(O.IC_CONSTANT_PV, ic) if x is o else x.set_initial_condition(O.IC_CONSTANT_PV, ic)
        x.set_perturbation(5, 0.02)
        x.initialize()
    return o, s


@pytest.mark.parametrize("ti", list(TI))
@pytest.mark.parametrize("nd,level,shape,mask", [(2, 9, (257, 1), True), (2, 5, (27, 19), False),
                                                 (3, 4, (1, 1, 1), True), (3, 5, (19, 9, 3), False)])
def test_masked_boxes_match_oracle(nd, level, shape, mask, ti):
    """257, 513, 1 and 513 cells: whole tiles and one cell more, and a cell
    that meets a ghost on every side."""
    o, s = _box(nd, level, shape, mask, ti)
    n = int(np.prod(shape))
    assert s.first_gc == o.first_gc == n and n % 256 == 1
    o.solve(6)
    s.solve(6)
    err = rel_l2(s.lhs, o.get("lhs"), nd)
    assert np.max(err) <= 1e-12, err
    assert abs(s.time() - o.time()) <= 1e-13 * o.time()


@pytest.mark.parametrize("bc", ["neumann", "dirichlet", "periodic"])
@pytest.mark.parametrize("grid", GRIDS)
def test_tiles_match_oracle(grid, bc):
    if bc == "periodic" and grid[2]:
        pytest.skip("periodic images are defined on uniform grids")
    for ti in TI:
        o, s = pair(*grid, ti, bc, "fp64")
        assert s.kernel() == "generic" and s.first_gc == o.first_gc
        o.solve(4)
        s.solve(4)
        n = o.first_gc
        err = rel_l2(s.lhs[:, :n], o.get("lhs")[:, :n], grid[0])
        assert np.max(err) <= 1e-12, (ti, err)
        # the ghosts hold the boundary conditions of the last step's start
        if n < s.ncells:
            g = rel_l2(s.lhs[:, n:], o.get("lhs")[:, n:], grid[0])
            assert np.max(g) <= 1e-12, (ti, g)
        assert abs(s.time() - o.time()) <= 1e-13 * o.time()
        s.close()


def test_tiles_fp32_state():
    o, s = pair(3, 4, 2, 0.25, 0.02, "ssp_rk3", "neumann", "fp32")
    o.solve(4)
    s.solve(4)
    n = o.first_gc
    err = rel_l2(s.lhs[:, :n], o.get("lhs")[:, :n], 3)
    # FP32 rounding (6e-8) of two stage states and of the fluxes per step
    assert 0 < np.max(err) <= 4 * 3 * 6e-8 * 8, err
    s.close()


def test_generic_forces_the_table_driven_kernel():
    """kernel="generic" runs the neighbour table's kernel on a refined grid,
    coarse/fine faces included, and kernel="tile" (auto's choice there) the
    tiles: the same states but for rounding, and not the same bits."""
    import hom3_amd as H
    _, s = pair(2, 4, 2, 0.2, 0.05, "ssp_rk3", "neumann", "fp64", kernel="auto")
    _, t = pair(2, 4, 2, 0.2, 0.05, "ssp_rk3", "neumann", "fp64", kernel="tile")
    for ti in TI:
        o, g = pair(2, 4, 2, 0.2, 0.05, ti, "dirichlet" if ti == "runge_kutta_2" else "neumann", "fp64",
                    kernel="generic")
        o.solve(4)
        g.solve(4)
        n = o.first_gc
        assert np.max(rel_l2(g.lhs[:, :n], o.get("lhs")[:, :n], 2)) <= 1e-12, ti
    s.solve(4)
    t.solve(4)
    np.testing.assert_array_equal(s.lhs, t.lhs)
    assert 0 < np.max(rel_l2(t.lhs[:, :n], g.lhs[:, :n], 2)) <= 1e-12
    # a periodic MUSCL solver has no tiles
    gr = H.Grid(2, [0.0] * 2, [1.0] * 2, 4)
    m = H.Solver(gr, physics="euler", time_integration="ssp_rk3", recon="muscl", kernel="tile")
    H.append_bcs(m, H.Periodic())
    with pytest.raises(RuntimeError, match="tile kernel requested"):
        m.build()
    with pytest.raises(RuntimeError, match="not built"):
        m.solve(1)


@pytest.mark.parametrize("nd,base", [(3, 4), (2, 6)])
def test_rounding_error_is_the_table_driven_kernels(nd, base):
    """The error after 60 SSP-RK3 steps from the same start against the same
    scheme in long double: on tiles as on the neighbour table.  It is a mean
    over 10^4 cells of independent roundings, so two orders of the same
    operations differ by some percent; 1.5 is far outside of that and below
    the factor of 3.7 that rounding the other product of U/3 + 2/3 s costs."""
    OL = O.long_double()
    o, s = pair(nd, base, 1, 0.2, 0.05, "ssp_rk3", "neumann", "fp64")
    _, g = pair(nd, base, 1, 0.2, 0.05, "ssp_rk3", "neumann", "fp64", kernel="generic")
    q0, n = o.get("lhs").copy(), o.first_gc
    og = OL.Grid(nd, [0.0] * nd, [1.0] * nd).min_level(base)
    og.refine_region(base + 1, OL.geom(OL.GEOM_SPHERE, [0.5, 0.4, 0.6][:nd], [0.2]), 0.05)
    og.balance()
    ol = OL.Solver(og, OL.phys(physics=OL.PHYS_EULER, nd=nd, ti=OL.TI_SSP_RK3, cfl=0.2))
    for geo in OL.cube_boundaries(nd, [0.0] * nd, [1.0] * nd):
        ol.append_bc(geo, OL.BC_EULER_NEUMANN, [])
    ol.set_ic(*((OL.IC_FOUR_QUADRANT, QUAD) if nd == 2 else (OL.IC_SPHERE, BALL)))
    ol.initialize()
    ol.set_lhs(q0)
    ol.set_time(0.0, 0.0, 0)
    ol.solve(60)
    exact = ol.get("lhs")[:, :n]
    err = []
    for x in (s, g):
        x.set_lhs(q0)
        x.reset_time(0.0, 0.0, 0)
        x.solve(60)
        err.append(np.sqrt(((x.lhs[:, :n] - exact) ** 2).sum() / (exact ** 2).sum()))
    print("cells", n, "error against long double: tiles", err[0], "table-driven", err[1])
    assert err[0] <= 1.5 * err[1], err


def test_fused_dt_equals_the_reduction():
    """The CFL bound fused into the last stage is the one a reduction over
    the new state gives."""
    _, s = pair(2, 4, 2, 0.2, 0.05, "ssp_rk3", "neumann", "fp64")
    s.solve(5)
    bound = s.min_dt()
    s.solve(1)
    assert s.dt() == bound
    _, a = pair(2, 4, 2, 0.2, 0.05, "ssp_rk3", "neumann", "fp64")
    a.solve(6)
    np.testing.assert_array_equal(a.lhs, s.lhs)


@pytest.mark.parametrize("kernel", ["tile", "generic", "auto"])
def test_fp32_state_does_not_depend_on_the_units(kernel):
    """The Euler equations do not change when density and pressure are scaled
    together, and a power of two changes no rounding: FP32 stage states at
    2^-80 (a gas of 1e-24) take the same steps as at 1.  kernel auto: the
    bricks of a uniform grid."""
    import hom3_amd as H
    args = (3, 4, 0, 0, 0) if kernel == "auto" else (3, 3, 1, 0.25, 0.1)
    _, s = pair(*args, "ssp_rk3", "neumann", "fp32", kernel=kernel)
    assert s.kernel() == ("brick" if kernel == "auto" else "generic")
    q0, n = s.lhs.copy(), s.first_gc
    out = []
    for scale in (1.0, 2.0 ** -80):
        s.set_lhs(q0 * scale)
        s.reset_time(0.0, 0.0, 0)
        s.solve(5)
        out.append((s.lhs[:, :n] / scale, s.time()))
    # (what underflows is 2^-46 of a term that it is added to)
    assert np.max(rel_l2(out[1][0], out[0][0], 3)) <= 1e-7
    assert abs(out[1][1] - out[0][1]) <= 1e-7 * out[0][1]
    if kernel != "tile":
        return
    b = []
    for scale in (1.0, 2.0 ** -80):
        s.set_lhs(q0 * scale)
        s.reset_time(0.0, 0.0, 0)
        B = H.Batch([s], "fp32")
        B.solve(5)
        b.append(B.state(0) / scale)
        B.close()
    assert np.max(rel_l2(b[1], b[0], 3)) <= 1e-7
