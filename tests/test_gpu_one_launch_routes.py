"""Which solves run as one kernel, and that the launches they are handed back to
return the same bits.

cfd_get_one_launch_counters says what ran; cfd_set_one_launch_bounds(arrive < 0)
takes the launches.  A route is given as (finished, handed back) of one solve:
one workgroup, several, the most rows or cells (finished); one more, which is
too large to be tried (neither); a halo that no workgroup holds (handed back).
"""
from __future__ import annotations

import threading
import time

import numpy as np
import pytest

import oracle_lib as O
from cfd_nssolver_forhpc_amd import capi, configs
from cfd_nssolver_forhpc_amd.solver import Simulation, uniform_grid

pytestmark = pytest.mark.gpu

RUNS, LARGE, BACK = (1, 0), (0, 0), (0, 1)


def make_sim(ncal):
    return Simulation(uniform_grid(ncal, (10.0, 6.0, 3.0)), configs.cylinder_params(100.0, 0.002, 2.5, 3.0, 1.0, 1e-10))


def delta(sim, before):
    return tuple(a - b for a, b in zip(sim.one_launch_counters(), before))[:2]


def bicg(sim, K):
    before = sim.one_launch_counters()
    sim.upload(capi.X, np.zeros(sim.N))
    it, _ = sim.bicgstab(tol=0.0, maxit=K)
    assert it == K
    return sim.download(capi.X), delta(sim, before)


def both_ways(sim, K, route):
    sim.one_launch_bounds(arrive=-1)
    want, way = bicg(sim, K)
    assert way == ((0, 0) if route == LARGE else BACK)
    assert np.isfinite(want).all()
    sim.one_launch_bounds()
    got, way = bicg(sim, K)
    assert way == route
    assert np.array_equal(got, want)


@pytest.mark.parametrize("ncal,K,route", [
    ((2, 2, 2), 1, RUNS), ((16, 16, 8), 20, RUNS), ((17, 11, 11), 20, RUNS), ((37, 25, 11), 20, RUNS),
    ((150, 75, 27), 10, RUNS), ((8, 8, 1000), 10, RUNS), ((64, 64, 128), 10, RUNS), ((64, 64, 129), 10, LARGE),
    ((16, 8, 4096), 5, RUNS)])
def test_bicgstab(require_gpu, ncal, K, route):
    print(f"one-launch route ncal={ncal} K={K}", flush=True)
    with make_sim(ncal) as sim:
        sim.init_state()
        sim.createPressureMatrix()
        b = np.random.default_rng(3).standard_normal(sim.N)
        sim.upload(capi.RHS, b - b.mean())
        both_ways(sim, K, route)


@pytest.mark.parametrize("ncal,route", [((24, 25, 10), RUNS), ((32, 32, 16), BACK)])
def test_uploaded_matrix_with_random_columns(require_gpu, ncal, route):
    with make_sim(ncal) as sim:
        sim.init_state()
        n = sim.N
        rng = np.random.default_rng(5)
        col = rng.integers(0, n, size=(7, n), dtype=np.int32)
        val = rng.uniform(-0.1, 0.1, size=(7, n))
        col[0], val[0] = np.arange(n), 1.0
        sim.set_ell(col, val)
        sim.upload(capi.RHS, rng.standard_normal(n))
        both_ways(sim, 4, route)


@pytest.mark.parametrize("ncal,route", [
    ((8, 6, 4), RUNS), ((9, 7, 5), RUNS), ((17, 11, 13), RUNS), ((64, 64, 64), RUNS), ((64, 64, 65), LARGE),
    ((8, 8, 1100), BACK)])
def test_sor_pipeline(require_gpu, ncal, route):
    print(f"one-launch SOR route ncal={ncal}", flush=True)
    grid = uniform_grid(ncal, (8.0, 6.0, 4.0))
    G = O.Grid(grid).G
    rng = np.random.default_rng(5)
    u1 = [1.0 + 0.05 * rng.standard_normal(G), 0.05 * rng.standard_normal(G), 0.05 * rng.standard_normal(G)]
    p0 = rng.standard_normal(G)
    prm = configs.cylinder_params(100.0, 0.002, 2.0, 1.0, 0.5, 1e-3)
    prm.solver = capi.CFD_SOLVER_SOR_PIPELINE
    with Simulation(grid, prm) as sim:
        sim.init_state()

        def sweeps(arrive):
            sim.one_launch_bounds(arrive=arrive)
            for c in range(3):
                sim.upload(capi.T1_U + c, u1[c])
            sim.upload(capi.P, p0)
            before = sim.one_launch_counters()
            it, err = sim.SorPipeLine(omega=1.8, crit=0.0, itmax=7)
            return sim.download(capi.P), it, err, delta(sim, before)

        want, it0, err0, way = sweeps(-1)
        assert way == ((0, 0) if route == LARGE else BACK)
        assert np.isfinite(want).all()
        got, it1, err1, way = sweeps(0)
        assert way == route
    assert (it1, err1) == (it0, err0)
    assert np.array_equal(got, want)


# a wait that runs out at once: every workgroup's, the first one's only (the
# others wait for a workgroup that has left)
@pytest.mark.parametrize("bounds", [dict(wait=1), dict(wait=512, wait_first=1)])
@pytest.mark.parametrize("ncal", [(17, 11, 11), (37, 25, 11), (64, 64, 16), (64, 64, 128)])
def test_bicgstab_whose_waits_run_out(require_gpu, ncal, bounds):
    print(f"one-launch waits ncal={ncal} {bounds}", flush=True)
    b = np.random.default_rng(3).standard_normal(int(np.prod(ncal)))
    b -= b.mean()
    got = []
    for lim in (dict(arrive=-1), bounds):
        with make_sim(ncal) as sim:
            sim.init_state()
            sim.createPressureMatrix()
            sim.upload(capi.X, np.zeros(sim.N))
            sim.one_launch_bounds(**lim)
            for k in range(12):  # from the last x; the restart rule starts at the tenth solve
                sim.upload(capi.RHS, (1.0 + 0.1 * k) * b)
                it, rel = sim.bicgstab(tol=1e-6, maxit=40)
            fin, back, _ = sim.one_launch_counters()
            assert fin + back == 12
            assert "wait_first" in lim or fin == 0  # a first workgroup may find every value at its first look
            got.append((sim.download(capi.X), it, rel, sim.solver_counters()))
    assert np.isfinite(got[0][0]).all()
    assert got[1][1:] == got[0][1:]
    assert np.array_equal(got[1][0], got[0][0])


def test_one_bound_for_a_workgroup(require_gpu):
    # The first workgroup leaves at once; each other one then has five waits an
    # iteration for words that do not come.  A poll took 0.21 us, so the first of
    # them takes 55 ms, the sums after it 1024 polls each and the halos 8192.
    with make_sim((64, 64, 16)) as sim:
        sim.init_state()
        sim.createPressureMatrix()
        sim.upload(capi.RHS, np.random.default_rng(3).standard_normal(sim.N))
        sim.upload(capi.X, np.zeros(sim.N))
        sim.one_launch_bounds(wait=1 << 18, wait_first=1)
        t = time.perf_counter()
        sim.bicgstab(tol=0.0, maxit=10)
        t = time.perf_counter() - t
        assert sim.one_launch_counters() == (0, 1, 1)
    assert t < 0.15  # three bounds, one for each sum of the iteration, are 165 ms


@pytest.mark.parametrize("bounds", [dict(wait=1), dict(wait=512, wait_first=1)])
def test_timesteps_whose_sweeps_run_out(require_gpu, bounds):
    grid = uniform_grid((33, 18, 12), (8.0, 6.0, 4.0))
    prm = configs.cylinder_params(100.0, 0.002, 2.0, 1.0, 0.5, 1e-3)
    prm.solver, prm.maxit = capi.CFD_SOLVER_SOR_PIPELINE, 60
    got = []
    for lim in (dict(arrive=-1), bounds):
        with Simulation(grid, prm) as sim:
            sim.setup(noise=1e-3, seed=1)
            sim.one_launch_bounds(**lim)
            steps = [sim.step().as_dict() for _ in range(3)]
            fin, back, _ = sim.one_launch_counters()
            assert fin + back == 8  # none in the first step, four in each that follows
            assert "wait_first" in lim or fin == 0
            got.append((steps, sim.download(capi.P), sim.download(capi.T0_U)))
    assert got[0][0] == got[1][0]
    assert np.isfinite(got[0][1]).all()
    assert np.array_equal(got[0][1], got[1][1]) and np.array_equal(got[0][2], got[1][2])


def test_launches_that_are_given_up(require_gpu):
    """An arrival bound of one poll: every try is given up, and tries get rarer."""
    with make_sim((37, 25, 11)) as sim:
        sim.init_state()
        sim.createPressureMatrix()
        b = np.random.default_rng(3).standard_normal(sim.N)
        sim.upload(capi.RHS, b - b.mean())
        sim.one_launch_bounds(arrive=-1)
        want, way = bicg(sim, 8)
        assert way == BACK
        sim.one_launch_bounds(arrive=1)
        before = sim.one_launch_counters()
        for _ in range(64):
            got, way = bicg(sim, 8)
            assert way == BACK
            assert np.array_equal(got, want)
        # the 1st, 3rd, 6th, 11th, 20th and 37th
        assert sim.one_launch_counters()[2] - before[2] == 6
        sim.one_launch_bounds()
        got, way = bicg(sim, 8)
        assert way == RUNS
        assert np.array_equal(got, want)


def test_contexts_on_two_threads(require_gpu):
    """Two systems of 256 workgroups each: one context's solves find the CUs
    taken while the other's hold them."""
    sims = [make_sim((64, 64, 128)) for _ in range(2)]
    try:
        want = []
        for k, sim in enumerate(sims):
            sim.init_state()
            sim.createPressureMatrix()
            b = np.random.default_rng(k).standard_normal(sim.N)
            sim.upload(capi.RHS, b - b.mean())
            sim.one_launch_bounds(arrive=-1)
            want.append(bicg(sim, 60)[0])
            sim.one_launch_bounds()
        before = [sim.one_launch_counters() for sim in sims]
        bad = []

        def work(k):
            for _ in range(20):
                if not np.array_equal(bicg(sims[k], 60)[0], want[k]):
                    bad.append(k)

        threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not bad
        for sim, b in zip(sims, before):
            fin, back = delta(sim, b)
            assert fin + back == 20
        print("finished, handed back, waited:", [sim.one_launch_counters() for sim in sims], flush=True)
    finally:
        for sim in sims:
            sim.close()
