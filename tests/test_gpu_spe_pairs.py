"""The SPE operator's kernels over pairs of columns (grids of 1024 tiles and
more, even nz) against the assembled operator with numpy: the product, to the
rounding of its seven terms, and four BiCGSTAB iterations from x = 0, to 1e-10
(as for the other forms).  A last walk of fewer tiles than the others and a
last tile of fewer planes; lines of 2 to 130 cells, with pairs past the line's
end in their tiles; walls, Dirichlet faces and joined z faces.
"""
from __future__ import annotations

import numpy as np
import pytest

from cfd_nssolver_forhpc_amd import capi, configs
from cfd_nssolver_forhpc_amd.solver import Simulation, uniform_grid
from test_gpu_krylov_folded import iterate, operator

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncal,periodic,pd", [
    ((67, 510, 34), 0, (0, 1, 0, 0, 0, 0)), ((130, 250, 18), 1, (0, 1, 0, 0, 0, 0)), ((64, 171, 130), 0, (1, 0, 0, 1, 1, 0)),
    ((515, 1000, 2), 0, (0, 0, 1, 0, 0, 1)), ((513, 130, 64), 1, (0, 1, 0, 0, 0, 0))])
def test_product_and_iterations(require_gpu, ncal, periodic, pd):
    print(f"SPE pairs case ncal={ncal} periodic={periodic} pd={pd}", flush=True)
    p = configs.cylinder_params(100.0, 0.002, 2.5, 3.0, 1.0, 1e-10)
    p.op, p.periodic_z = capi.CFD_OP_SPE, periodic
    for f in range(6):
        p.p_dirichlet[f] = pd[f]
    with Simulation(uniform_grid(ncal, (10.0, 6.0, 3.0)), p) as sim:
        sim.init_state()
        sim.createPressureMatrix()
        sim.setupPressure()
        A = operator(sim, capi.CFD_OP_ELL)
        rng = np.random.default_rng(8)
        x, b = rng.standard_normal(sim.N), rng.standard_normal(sim.N)
        sim.upload(capi.X, x)
        sim.spmv(op=capi.CFD_OP_SPE)
        # rows sum to 2 at most in absolute value; entries and terms are rounded a dozen times
        assert np.abs(sim.download(capi.VEC_A) - A(x)).max() <= 24 * np.finfo(float).eps * np.abs(x).max()
        sim.upload(capi.RHS, b)
        sim.time_kernel(4, 3)
        got, want = sim.download(capi.VEC_B), iterate(A, b, 4)
        assert np.linalg.norm(got - want) < 1e-10 * np.linalg.norm(want)
