"""BiCGSTAB iterations of the launch path around the sizes where its
reductions move into the updates that use them (at most 1024 partials of every
dot; at most 4096 of the first one; none), against the iteration written with
numpy: four iterations from x = 0 on a random right-hand side, to 1e-10 of x
(sums of 2.3 million terms differ by 1e-13, grown by four iterations of a
residual that is still of order one), and a whole solve's count and residual.
"""
from __future__ import annotations

import numpy as np
import pytest

from cfd_nssolver_forhpc_amd import capi, configs
from cfd_nssolver_forhpc_amd.solver import Simulation, uniform_grid

pytestmark = pytest.mark.gpu


def make(ncal, op):
    p = configs.cylinder_params(100.0, 0.002, 2.5, 3.0, 1.0, 1e-10)
    p.op = op
    sim = Simulation(uniform_grid(ncal, (10.0, 6.0, 3.0)), p)
    sim.init_state()
    sim.createPressureMatrix()
    if op == capi.CFD_OP_SPE:
        sim.setupPressure()
    if op == capi.CFD_OP_CSR:
        sim.createPressureMatrixCSR()
    return sim


def operator(sim, op):
    if op == capi.CFD_OP_CSR:  # closes every face (the builder's rule), so not the ELL operator
        ptr, ci, cv = sim.csr()
        return lambda x: np.add.reduceat(cv * x[ci], ptr[:-1])
    col, val = (q.reshape(7, -1) for q in sim.ell())
    return lambda x: sum(v * x[c] for c, v in zip(col, val))


def iterate(A, b, n):
    x, r = np.zeros_like(b), b.copy()
    r0, p, rho = r.copy(), r.copy(), r @ r
    for _ in range(n):
        ap = A(p)
        alpha = rho / (ap @ r0)
        s = r - alpha * ap
        as_ = A(s)
        omega = (as_ @ s) / (as_ @ as_)
        x += alpha * p + omega * s
        r = s - omega * as_
        rho, pre = r @ r0, rho
        p = r + (alpha / omega) * (rho / pre) * (p - omega * ap)
    return x


@pytest.mark.parametrize("ncal,op", [
    ((16, 12, 10), capi.CFD_OP_SPE), ((33, 17, 9), capi.CFD_OP_CSR), ((64, 32, 32), capi.CFD_OP_SPE),
    ((128, 64, 64), capi.CFD_OP_CSR), ((128, 64, 65), capi.CFD_OP_ELL), ((128, 96, 85), capi.CFD_OP_SPE),
    ((128, 128, 64), capi.CFD_OP_ELL), ((101, 99, 105), capi.CFD_OP_ELL), ((128, 128, 128), capi.CFD_OP_ELL),
    ((150, 127, 111), capi.CFD_OP_ELL), ((150, 127, 111), capi.CFD_OP_SPE)])
def test_iterations_against_numpy(require_gpu, ncal, op):
    print(f"folded case ncal={ncal} op={op}", flush=True)
    with make(ncal, op) as sim:
        A = operator(sim, op)
        b = np.random.default_rng(9).standard_normal(sim.N)
        sim.upload(capi.RHS, b)
        sim.time_kernel(4, 3)
        got, want = sim.download(capi.VEC_B), iterate(A, b, 4)
        assert np.linalg.norm(got - want) < 1e-10 * np.linalg.norm(want)


@pytest.mark.parametrize("ncal,op,pc", [((24, 20, 16), capi.CFD_OP_SPE, False), ((40, 33, 21), capi.CFD_OP_CSR, False),
                                        ((128, 64, 65), capi.CFD_OP_ELL, True), ((48, 32, 24), capi.CFD_OP_SPE, True)])
def test_stops_where_the_residual_says(require_gpu, ncal, op, pc):
    with make(ncal, op) as sim:
        A = operator(sim, op)
        b = A(np.random.default_rng(10).standard_normal(sim.N))
        p = sim.params
        if pc:
            p.precond = capi.CFD_PRECOND_MG
            sim.set_params(p)

        def solve(maxit):
            p.maxit, p.tol = maxit, 1e-6
            sim.set_params(p)
            sim.upload(capi.RHS, b)
            sim.upload(capi.X, np.zeros(sim.N))
            it, rel = sim.solve()
            y = sim.download(capi.X)
            res = np.linalg.norm(b - A(y)) / np.linalg.norm(b)
            assert abs(res - rel) < 1e-3 * rel + 1e-12
            return it, rel

        it, rel = solve(2000)
        assert it > 1 and rel < 1e-6
        n, r = solve(it - 1)  # stopped by the cap
        assert n == it - 1 and r >= 1e-6
        assert solve(it) == (it, rel)
