"""Data-flow kernels beside other work on the GPU: the switch that turns them
off, whose wait timed out, cooperative launches, and several solvers at once."""
import threading

import numpy as np
import pytest

from spgrid_topo_opt_amd import _lib
from spgrid_topo_opt_amd import workloads as W

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.fixture(scope="module")
def box45():
    """45x23x19 cells, 3 levels: level 0 and the explicit level 2 sweep by data flow"""
    return _lib.Solver(W.box(45, 23, 19, seed=6, mg_levels=3))


@pytest.fixture(scope="module")
def box96():
    """96x60x60 cells, 4 levels: the explicit level 2 has 24x15x15 cells"""
    return _lib.Solver(W.box(96, 60, 60, seed=6, mg_levels=4))


def sweep(s, level, **kw):
    n = len(s.level_nodes(level)[0])
    rng = np.random.default_rng(17)
    u, b = rng.standard_normal((n, 3)) * 1e-3, rng.standard_normal((n, 3))
    return s.kernel(_lib.OP_GS_SWEEP, level, u, b, **kw)


@pytest.mark.parametrize("box,level,name", [("box45", 0, "level-0 sweep"), ("box96", 2, "sweep of an explicit level")])
def test_a_time_out_names_its_kernel(box, level, name, request, monkeypatch):
    """a wait cut to one wall-clock tick (set from the host) ends the kernel; a
    wait that is over within two loads does not notice, so a few sweeps"""
    s = request.getfixturevalue(box)
    monkeypatch.setenv("SPG_COOP_LIMIT_TICKS", "1")
    with pytest.raises(_lib.SpgError, match=name + ": a wait timed out"):
        for _ in range(50):
            sweep(s, level)
    monkeypatch.delenv("SPG_COOP_LIMIT_TICKS")
    sweep(s, level)


@pytest.mark.parametrize("level", [0, 2])
def test_one_switch_turns_all_data_flow_kernels_off(box45, level, monkeypatch):
    """SPG_DATA_FLOW=0: nothing waits, so a one-tick limit ends nothing, in
    sweeps and boundary phases; results to 1e-12 of the data-flow ones (FP64)"""
    n = len(box45.level_nodes(level)[0])
    b = np.random.default_rng(3).standard_normal((n, 3))

    def phase(sweeps):  # 3 is the map's sweep count on small sets
        return box45.kernel(_lib.OP_GS_BOUNDARY, level, np.zeros((n, 3)), b, sweeps=sweeps)

    want = sweep(box45, level), phase(3), phase(2)
    monkeypatch.setenv("SPG_DATA_FLOW", "0")
    monkeypatch.setenv("SPG_COOP_LIMIT_TICKS", "1")
    got = sweep(box45, level), phase(3), phase(2)
    for g, w in zip(got, want):
        assert rel(g, w) < 1e-12


@pytest.mark.parametrize("prec,tol", [(1, 1e-13), (0, 1e-6)])
@pytest.mark.parametrize("level", [0, 2])
def test_cooperative_launches_cover_the_sweeps(box45, level, prec, tol, monkeypatch):
    want = sweep(box45, level, precision=prec)
    monkeypatch.setenv("SPG_COOP_LAUNCH", "1")
    for fwd in (True, False):
        monkeypatch.setenv("SPG_COOP_LAUNCH", "1")
        got = sweep(box45, level, precision=prec, forward=fwd)
        monkeypatch.setenv("SPG_COOP_LAUNCH", "0")
        assert rel(got, sweep(box45, level, precision=prec, forward=fwd)) < tol
    assert np.isfinite(want).all()


@pytest.mark.parametrize("coop", ["0", "1"])
def test_solvers_on_several_threads(coop, monkeypatch, capfd):
    """four solvers of up to 4,000 blocks solve at the same time, three times
    each, in both precisions: solutions as alone, and no wait times out"""
    monkeypatch.setenv("SPG_COOP_LAUNCH", coop)
    probs = [W.box(64, 43, 43, seed=1, mg_levels=3), W.box(64, 43, 43, seed=2, mg_levels=3),
             W.box(96, 50, 40, seed=3, mg_levels=4), W.box(45, 23, 19, seed=4, mg_levels=3)]
    solvers = [_lib.Solver(p) for p in probs]

    def both(s):
        return (s.solve(tolerance=1e-10, precision=1)[0], s.solve_mixed(tolerance=1e-8)[0])

    alone = [both(s) for s in solvers]
    got, errors = [[] for _ in solvers], []

    def work(i):
        try:
            for _ in range(3):
                got[i].append(both(solvers[i]))
        except Exception as e:  # reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(solvers))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for g, w in zip(got, alone):
        assert len(g) == 3
        for pair in g:
            # FP64 solves to 1e-10 and mixed ones to 1e-8 of the residual
            assert rel(pair[0][..., :3], w[0][..., :3]) < 1e-8
            assert rel(pair[1][..., :3], w[1][..., :3]) < 1e-5
    assert "timed out" not in capfd.readouterr().err
    for s in solvers:
        s.close()


@pytest.mark.parametrize("shape,levels,level", [((45, 23, 19), 3, 0), ((24, 40, 40), 4, 2)])
def test_dense_maps_that_get_no_memory(shape, levels, level, monkeypatch):
    """the maps refused at creation: the solver is created without them, its
    boundary phases (of the level's own sweep count) run by data flow, solves
    reach the same solution, also after a density update"""
    p = W.box(*shape, seed=5, mg_levels=levels)
    with_maps = _lib.Solver(p)
    monkeypatch.setenv("SPG_MAP_MAX_MB", "0")
    s = _lib.Solver(p)
    monkeypatch.delenv("SPG_MAP_MAX_MB")
    # two maps in FP64 and FP32 of at least this level's set
    gx, gf = s.level_nodes(level)
    assert with_maps.info()["hbm_bytes"] - s.info()["hbm_bytes"] > 10e6
    rng = np.random.default_rng(11)
    u, b = rng.standard_normal((len(gx), 3)) * 1e-3, rng.standard_normal((len(gx), 3))
    u[(gf & 1) == 0] = 0
    for prec, tol in ((1, 1e-11), (0, 1e-4)):
        want = with_maps.kernel(_lib.OP_GS_BOUNDARY, level, u, b, precision=prec, sweeps=3)
        assert rel(s.kernel(_lib.OP_GS_BOUNDARY, level, u, b, precision=prec, sweeps=3), want) < tol
    for density in (p.density, p.density * 0.9):
        for x in (s, with_maps):
            x.update_density(density)
        want, got = (x.solve(tolerance=1e-10, precision=1)[0] for x in (with_maps, s))
        assert rel(got[..., :3], want[..., :3]) < 1e-8
    s.close()
    with_maps.close()
