"""The SPE product between cfd_set_params and the next set-up: the diagonal is
that of the boundary conditions it was set up with, the z neighbours across the
seam those of the parameters now, on grids of 1024 tiles and more (where the
diagonal is formed again) and fewer (where it is read).

Tolerance: a row's entries sum to 3 at most in absolute value, and its terms are
rounded a dozen times.
"""
from __future__ import annotations

import numpy as np
import pytest

from cfd_nssolver_forhpc_amd import capi, configs
from cfd_nssolver_forhpc_amd.solver import Simulation, uniform_grid

pytestmark = pytest.mark.gpu

WALLS, OPEN = (0, 0, 0, 0, 0, 0), (0, 1, 1, 0, 1, 1)


def product(grid, set_up, now, x):
    per0, pd = set_up
    n = grid.ncal
    D, Ds = (grid.Dx, grid.Dy, grid.Dz), (grid.Dxs, grid.Dys, grid.Dzs)
    x = x.reshape(n)
    diag, off = 0.0, 0.0
    for a in range(3):
        shape = [1, 1, 1]
        shape[a] = n[a]
        w = D[a][2:n[a] + 2]
        cm, cp = 1.0 / w / Ds[a][1:n[a] + 1], 1.0 / w / Ds[a][2:n[a] + 2]
        dm, dp, om, op = cm.copy(), cp.copy(), cm.copy(), cp.copy()
        if not (a == 2 and per0):
            dm[0] *= pd[2 * a]
            dp[-1] *= pd[2 * a + 1]
        if not (a == 2 and now):
            om[0] = op[-1] = 0.0
        diag = diag + (dm + dp).reshape(shape)
        off = off + om.reshape(shape) * np.roll(x, 1, a) + op.reshape(shape) * np.roll(x, -1, a)
    return (x - off / diag).ravel()


@pytest.mark.parametrize("ncal", [(67, 510, 34), (40, 33, 18)])
@pytest.mark.parametrize("set_up,now", [((1, OPEN[:4] + (0, 0)), 0), ((0, WALLS), 1), ((0, OPEN), 0)])
def test_product_after_set_params(require_gpu, ncal, set_up, now):
    grid = uniform_grid(ncal, (10.0, 6.0, 3.0))
    p = configs.cylinder_params(100.0, 0.002, 2.5, 3.0, 1.0, 1e-10)
    p.op, p.periodic_z = capi.CFD_OP_SPE, set_up[0]
    for f in range(6):
        p.p_dirichlet[f] = set_up[1][f]
    with Simulation(grid, p) as sim:
        sim.init_state()
        sim.createPressureMatrix()
        sim.setupPressure()
        p.periodic_z = now
        for f in range(6):
            p.p_dirichlet[f] = 1 - set_up[1][f] if f < 4 else 0
        sim.set_params(p)
        x = np.random.default_rng(8).standard_normal(sim.N)
        sim.upload(capi.X, x)
        sim.spmv(op=capi.CFD_OP_SPE)
        want = product(grid, set_up, now, x)
        assert np.abs(sim.download(capi.VEC_A) - want).max() <= 36 * np.finfo(float).eps * np.abs(x).max()
