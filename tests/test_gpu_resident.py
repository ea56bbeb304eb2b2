"""The one-launch BiCGSTAB of small ELL systems against the launch path.

cfd_time_kernel(4) runs the launch path's iterations (eight kernels each, no
stop test) on scratch vectors from x = 0, so after K + 1 of them VEC_B holds
what cfd_bicgstab(tol = 0, maxit = K) must return, bit for bit: both sum in the
same order.  Sizes: one workgroup (N <= 2048), an odd and an even number of
1024-row groups (their sums cross workgroups differently), a ragged end, the
largest halo (lines longer than a workgroup's 512 rows), the largest resident
system and the next, and a solve that takes more than one launch; random
columns, whose halo fits the workgroup or does not (the launch path).
"""
from __future__ import annotations

import numpy as np
import pytest

from cfd_nssolver_forhpc_amd import capi, configs
from cfd_nssolver_forhpc_amd.solver import Simulation, uniform_grid

pytestmark = pytest.mark.gpu


def make_sim(ncal):
    return Simulation(uniform_grid(ncal, (10.0, 6.0, 3.0)), configs.cylinder_params(100.0, 0.002, 2.5, 3.0, 1.0, 1e-10))


def launch_path(sim, K):
    """x after K + 1 launched iterations from x = 0 (one warm-up, K timed)."""
    sim.time_kernel(4, K)
    return sim.download(capi.VEC_B)


def zero_mean(n, seed):
    b = np.random.default_rng(seed).standard_normal(n)
    return b - b.mean()


@pytest.mark.parametrize("ncal,K", [((2, 2, 2), 3), ((8, 8, 8), 20), ((16, 16, 8), 25), ((17, 11, 11), 25),
                                    ((33, 17, 9), 40), ((32, 16, 8), 40), ((37, 25, 11), 30), ((128, 64, 4), 60),
                                    ((150, 75, 27), 30), ((8, 8, 1000), 20),
                                    ((64, 64, 128), 20), ((64, 64, 129), 20)])
def test_same_bits_as_the_launch_path(require_gpu, ncal, K):
    print(f"resident case ncal={ncal} K={K}", flush=True)
    with make_sim(ncal) as sim:
        sim.init_state()
        sim.createPressureMatrix()
        sim.upload(capi.RHS, zero_mean(sim.N, 3))
        want = launch_path(sim, K)
        sim.upload(capi.X, np.zeros(sim.N))
        it, _ = sim.bicgstab(tol=0.0, maxit=K)
        assert it == K
        assert np.array_equal(sim.download(capi.X), want, equal_nan=True)


def test_more_iterations_than_a_launch(require_gpu):
    K = 4200
    with make_sim((150, 75, 27)) as sim:
        sim.init_state()
        sim.createPressureMatrix()
        sim.upload(capi.RHS, zero_mean(sim.N, 4))
        want = launch_path(sim, K)
        assert np.isfinite(want).all()
        sim.upload(capi.X, np.zeros(sim.N))
        it, _ = sim.bicgstab(tol=0.0, maxit=K)
        assert it == K
        assert np.array_equal(sim.download(capi.X), want)


@pytest.mark.parametrize("ncal", [(24, 25, 10), (32, 32, 16)])  # the halo of random columns fits; does not
def test_matrix_that_is_no_stencil(require_gpu, ncal):
    with make_sim(ncal) as sim:
        sim.init_state()
        n = sim.N
        rng = np.random.default_rng(5)
        col = rng.integers(0, n, size=(7, n), dtype=np.int32)
        val = rng.uniform(-0.1, 0.1, size=(7, n))
        col[0], val[0] = np.arange(n), 1.0
        sim.set_ell(col, val)
        b = zero_mean(n, 6)
        sim.upload(capi.RHS, b)
        want = launch_path(sim, 4)
        sim.upload(capi.X, np.zeros(n))
        sim.bicgstab(tol=0.0, maxit=4)
        assert np.array_equal(sim.download(capi.X), want)
        sim.upload(capi.X, np.zeros(n))
        it, rel = sim.bicgstab(tol=1e-10, maxit=500)
        x = sim.download(capi.X)
        assert rel < 1e-10
        # the recursive residual is the true one to rounding: 1e-10 and
        # a few hundred roundings of O(1) values
        assert np.linalg.norm(b - (val * x[col]).sum(axis=0)) <= 1.1e-10 * np.linalg.norm(b) + 1e-13 * np.linalg.norm(x)
