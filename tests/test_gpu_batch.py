"""Batched instances (one persistent kernel per RK stage, hipGraph steps,
autotuned launch shape) against the oracle, instance by instance.  Each
instance is an independent first-order Euler solver with its own 2:1
refined grid, dt, time and step (solver.hpp:140-145 per instance)."""
import numpy as np
import pytest

import oracle as O
from tests.scenarios import rel_l2

pytestmark = pytest.mark.gpu

TI = {"euler_forward": O.TI_EULER_FWD, "runge_kutta_2": O.TI_HEUN_RK2, "ssp_rk3": O.TI_SSP_RK3}


def oracle_instance(prm, ti, cfl):
    g = O.Grid(2, [0.0, 0.0], [1.0, 1.0]).min_level(prm["level"])
    if prm["extra"] > 0:
        half = 0.5 * prm["radius"]
        g.refine_region(prm["level"] + prm["extra"], O.geom(O.GEOM_SPHERE, prm["centre"], [half]), half)
        g.balance()
    s = O.Solver(g, O.phys(physics=O.PHYS_EULER, nd=2, ti=TI[ti], cfl=cfl))
    s.append_cube_bcs([O.BC_EULER_NEUMANN] * 4)
    s.set_ic(O.IC_FOUR_QUADRANT, prm["ic"])
    s.initialize()
    return g, s


def make(seed, n, ti, cfl=0.4, levels=(3, 4, 5)):
    import hom3_amd as H
    from hom3_amd.batch import build_instance
    prms = H.four_quadrant_instances(seed, n, levels=levels)
    gpu = [build_instance(H, p, ti=ti, cfl=cfl) for p in prms]
    ora = [oracle_instance(p, ti, cfl) for p in prms]
    return prms, gpu, ora


@pytest.mark.parametrize("ti,graph", [("ssp_rk3", True), ("ssp_rk3", False), ("runge_kutta_2", True),
                                      ("euler_forward", True)])
def test_batch_matches_oracle(ti, graph):
    import hom3_amd as H
    prms, gpu, ora = make(11, 6, ti)
    assert any(p["extra"] > 0 for p in prms) and len({p["level"] for p in prms}) > 1
    B = H.Batch(gpu, "fp64")
    nsteps = 5
    B.solve(2, graph=graph)
    B.solve(nsteps - 2, graph=graph)
    for i, (g, o) in enumerate(ora):
        o.solve(nsteps)
        n = o.first_gc
        err = rel_l2(B.state(i), o.get("lhs")[:, :n], 2)
        assert np.max(err) <= 1e-12, (i, err)
        t, dt, st = B.time(i)
        assert st == nsteps
        assert abs(t - o.time()) <= 1e-13 * o.time()
        assert abs(dt - o.dt()) <= 1e-13 * o.dt()
        # the source solver is left unchanged
        assert gpu[i].step() == 0
    B.close()


def test_batch_of_one_equals_solver():
    import hom3_amd as H
    from hom3_amd.batch import build_instance
    prms, gpu, ora = make(3, 1, "ssp_rk3")
    B = H.Batch(gpu, "fp64")
    B.solve(4)
    # same steps; the tiles' AUSM differs from the table-driven solver
    # kernel only in rounding (primitives computed once per cell)
    table = build_instance(H, prms[0], ti="ssp_rk3", cfl=0.4, kernel="generic")
    table.solve(4)
    err = rel_l2(B.state(0), table.lhs[:, :table.first_gc], 2)
    assert np.max(err) <= 1e-13, err
    assert B.time(0)[2] == table.step() == 4
    # the solver on tiles runs the batch's kernel on the same lists
    tiles = build_instance(H, prms[0], ti="ssp_rk3", cfl=0.4, kernel="tile")
    tiles.solve(4)
    np.testing.assert_array_equal(B.state(0), tiles.lhs[:, :tiles.first_gc])
    B.close()


def test_autotune_and_configs_do_not_change_results():
    import hom3_amd as H
    prms, gpu, ora = make(5, 5, "ssp_rk3")
    B1 = H.Batch(gpu, "fp64")
    choice = B1.autotune()
    assert choice["block"] in (128, 256, 512) and choice["stage_ms"] > 0
    B1.solve(3)
    B2 = H.Batch(gpu, "fp64")
    B2.set_config(64, 64, 7)
    B2.solve(3, graph=False)
    for i in range(len(gpu)):
        np.testing.assert_array_equal(B1.state(i), B2.state(i))
    B1.close()
    B2.close()


def test_config_reports_what_runs():
    import hom3_amd as H
    prms, gpu, ora = make(5, 5, "ssp_rk3")
    B = H.Batch(gpu, "fp64")
    items = sum(-(-s.first_gc // 256) for s in gpu)
    c = B.config()
    assert (c["block"], c["tile"], c["items"]) == (256, 256, items) and c["grid"] >= 1
    B.set_config(64, 64, 7)
    assert B.config() == dict(block=256, tile=256, grid=7, items=items)
    for bad in ((63, 256, 1), (1024, 1024, 1), (256, 128, 1), (256, 256, 0)):
        with pytest.raises(RuntimeError):
            B.set_config(*bad)
    a = B.autotune()
    assert B.config() == dict(block=256, tile=256, grid=a["grid"], items=items)
    B.close()


def test_batch_fp32_state_error():
    """FP32 stage buffers and flux arithmetic, FP64 U^n and accumulation:
    relative L2 error against the FP64 oracle stays below 1e-5."""
    import hom3_amd as H
    prms, gpu, ora = make(17, 4, "ssp_rk3")
    B = H.Batch(gpu, "fp32")
    B.solve(5)
    for i, (g, o) in enumerate(ora):
        o.solve(5)
        err = rel_l2(B.state(i), o.get("lhs")[:, :o.first_gc], 2)
        assert np.max(err) <= 1e-5, (i, err)
        assert np.max(err) > 0
    B.close()
