"""The assembled ELL operator, whose entries the kernels form again from the
axis coefficients, against the same matrix downloaded and uploaded, whose
stored entries they read: the products, the launch path's iterations and the
V-cycle-preconditioned ones are equal bit for bit.

Sizes: row-wise kernels (a plane no multiple of the block's threads), planes in
blocks of 512 and of 256 rows with a last block of fewer than four planes, more
planes than a period (a thread of the row-wise kernel takes several rows), two
planes, lines of two cells, z faces joined, walls and Dirichlet faces, uneven
spacing.
"""
from __future__ import annotations

import numpy as np
import pytest

from cfd_nssolver_forhpc_amd import capi, configs
from cfd_nssolver_forhpc_amd.solver import GridArrays, Simulation, axis_tanh, axis_uniform

pytestmark = pytest.mark.gpu

CASES = [((37, 25, 11), 0, (0, 1, 0, 0, 0, 0)), ((5, 32, 16), 0, (0, 0, 0, 0, 0, 0)), ((6, 32, 24), 1, (0, 1, 0, 0, 0, 0)),
         ((8, 64, 8), 0, (1, 0, 0, 1, 1, 0)), ((2, 128, 4), 1, (0, 1, 0, 0, 0, 0)), ((9, 512, 2), 0, (0, 0, 1, 0, 0, 1)),
         ((16, 16, 32), 1, (0, 1, 0, 0, 0, 0)), ((37, 1024, 512), 0, (0, 1, 0, 0, 0, 0))]


@pytest.mark.parametrize("ncal,periodic,pd", CASES)
def test_same_bits_as_the_stored_entries(require_gpu, ncal, periodic, pd):
    print(f"grid ELL case ncal={ncal} periodic={periodic} pd={pd}", flush=True)
    big = ncal[0] * ncal[1] * ncal[2] > 10**7
    p = configs.cylinder_params(100.0, 0.002, 2.5, 3.0, 1.0, 1e-10)
    p.periodic_z = periodic
    for f in range(6):
        p.p_dirichlet[f] = pd[f]
    p.precond, p.mg_nu, p.maxit = capi.CFD_PRECOND_MG, 1, 2
    y = axis_tanh(ncal[1], 6.0, 3.0, 0.01, 1.0, 1.05) if ncal[1] == 64 else axis_uniform(ncal[1], 6.0)
    ax = [axis_uniform(ncal[0], 10.0), y, axis_uniform(ncal[2], 3.0)]
    with Simulation(GridArrays(ncal, *[a[q] for q in range(3) for a in ax], 10.0, 6.0, 3.0), p) as sim:
        sim.init_state()
        sim.createPressureMatrix()
        rng = np.random.default_rng(7)
        x, b = rng.standard_normal(sim.N), rng.standard_normal(sim.N)

        def outputs():
            out = []
            sim.upload(capi.X, x)
            sim.spmv()
            out.append(sim.download(capi.VEC_A))
            sim.upload(capi.RHS, b)
            sim.time_kernel(4, 3)
            out.append(sim.download(capi.VEC_B))
            sim.upload(capi.X, np.zeros(sim.N))
            if not big:
                sim.solve()
                out.append(sim.download(capi.X))
            return out

        got = outputs()
        sim.set_ell(*sim.ell())
        want = outputs()
        for q, (g, w) in enumerate(zip(got, want)):
            assert np.isfinite(w).all(), q
            assert np.array_equal(g, w), q
        sim.createPressureMatrix()  # the grid's own operator again
        assert np.array_equal(outputs()[1], want[1])
