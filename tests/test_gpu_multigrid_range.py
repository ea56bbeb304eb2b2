"""The FP32 V-cycle near the ends of FP32's exponent range.

Scaling every length by a power of two scales the Laplacian and the right-hand
side r / jp by another and leaves the preconditioned iteration's x as it was,
bit for bit, while nothing overflows or goes below the normal numbers inside a
cycle.  With cells 2^-62 long the diagonals are 6 x 2^124 (their reciprocals are
not normal), with 2^66 they are 6 x 2^-132 (not normal themselves).  The grid has
fused passes on its finest level, and its coarsest is swept in registers.
"""
from __future__ import annotations

import numpy as np
import pytest

from cfd_nssolver_forhpc_amd import capi, configs
from cfd_nssolver_forhpc_amd.solver import Simulation, uniform_grid

pytestmark = pytest.mark.gpu


def two_iterations(h, amplitude):
    ncal = (50, 26, 10)
    p = configs.cylinder_params(100.0, 0.002, 1.0, 1.0, 1.0, 1e-30)
    p.precond, p.mg_nu, p.maxit = capi.CFD_PRECOND_MG, 4, 1
    p.precision, p.mixed_mode = capi.CFD_MIXED, capi.CFD_MIXED_PC32
    with Simulation(uniform_grid(ncal, tuple(h * n for n in ncal)), p) as sim:
        sim.init_state()
        sim.createPressureMatrix()
        b = np.random.default_rng(11).standard_normal(sim.N)
        sim.upload(capi.RHS, amplitude * (b - b.mean()))
        sim.upload(capi.X, np.zeros(sim.N))
        it, _ = sim.solve()
        assert it == 1
        return sim.download(capi.X)


@pytest.mark.parametrize("exponent,amplitude", [(-62, 2.0 ** -8), (66, 2.0 ** 40)])
def test_scaled_lengths(require_gpu, exponent, amplitude):
    want = two_iterations(1.0, amplitude)
    assert np.isfinite(want).all() and np.abs(want).max() > 0.0
    assert np.array_equal(two_iterations(2.0 ** exponent, amplitude), want)
