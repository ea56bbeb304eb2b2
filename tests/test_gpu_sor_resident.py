"""SorPipeLine's sweeps in one launch, and the launches that take over where a
grid does not fit, bit for bit against the oracle's red-black restatement.

Sizes: one workgroup and two; odd nz; the most cells, and past them (launches
that fold their maxima, at most 1024 blocks, and that do not); lines whose halo
no workgroup holds; more sweeps than a launch; a stop by the criterion; one
sweep.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from cfd_nssolver_forhpc_amd import capi, configs
from cfd_nssolver_forhpc_amd.solver import Simulation, uniform_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncal,crit,itmax", [
    ((8, 6, 4), 0.0, 9), ((16, 8, 8), 0.0, 9), ((9, 7, 5), 0.0, 8), ((17, 11, 13), 0.0, 7), ((64, 64, 64), 0.0, 6),
    ((64, 64, 65), 0.0, 6), ((128, 64, 64), 0.0, 6), ((128, 64, 65), 0.0, 5), ((8, 8, 1100), 0.0, 6),
    ((16, 12, 10), 0.0, 4200), ((40, 20, 11), 1e-6, 5000), ((24, 20, 16), 0.0, 1)])
def test_same_bits_as_the_oracle(require_gpu, ncal, crit, itmax):
    print(f"resident SOR case ncal={ncal} crit={crit} itmax={itmax}", flush=True)
    grid = uniform_grid(ncal, (8.0, 6.0, 4.0))
    g = O.Grid(grid)
    rng = np.random.default_rng(5)
    u1 = [1.0 + 0.05 * rng.standard_normal(g.G), 0.05 * rng.standard_normal(g.G), 0.05 * rng.standard_normal(g.G)]
    p0 = rng.standard_normal(g.G)
    prm = configs.cylinder_params(100.0, 0.002, 2.0, 1.0, 0.5, crit)
    prm.solver = capi.CFD_SOLVER_SOR_PIPELINE
    with Simulation(grid, prm) as sim:
        sim.init_state()
        for c in range(3):
            sim.upload(capi.T1_U + c, u1[c])
        sim.upload(capi.P, p0)
        it, err = sim.SorPipeLine(omega=1.8, crit=crit, itmax=itmax)
        got = sim.download(capi.P)
    p = p0.copy()
    oit = C.c_int()
    oerr = O.lib().orc_sor_rb_vw(g.ref, 0.002, 1.8, crit, itmax, *u1, p, C.byref(oit))
    assert it == oit.value and err == oerr
    assert np.array_equal(got, p)
