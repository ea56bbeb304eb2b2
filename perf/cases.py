"""The work this library is used for, as cases that can be timed.

A case is a short job through the public entry points: a run of
prediction-correction timesteps from a seeded initial state, a pressure solve
on a right-hand side that the caller supplies, a solve on the caller's own
device buffers, or an objective run with its discrete adjoint.  Where the
context holds the fields on the device, a pass ends as a user's program does,
by fetching them into host buffers that it allocated once (pinned).

  listed()   the cases, from the smallest grid of the tests to the largest workload
  draw(rng)  another case of the same ranges
  prepare()  grid, context, operator and seeded inputs
  run()      one pass; it starts from the prepared inputs, so it can be repeated
  work()     bytes and operations that a pass cannot do without
  exact()    the solution of a converged pressure solve, by diagonalising the
             operator's three axes in FP64 with torch
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from cfd_nssolver_forhpc_amd import adjoint, capi, configs, solver

OPS = {"ELL": capi.CFD_OP_ELL, "SPE": capi.CFD_OP_SPE, "CSR": capi.CFD_OP_CSR}
CONV = {"QUICK": capi.CFD_CONV_QUICK, "LUD": capi.CFD_CONV_LUD, "UD": capi.CFD_CONV_UD}
SOLVERS = {"BICGSTAB": capi.CFD_SOLVER_BICGSTAB, "RBSOR": capi.CFD_SOLVER_RBSOR,
           "SOR_PIPELINE": capi.CFD_SOLVER_SOR_PIPELINE}


def _case(kind, nx, ny, nz, **over):
    """kind: "run" (timesteps), "poisson" (a pressure solve in a context),
    "device" (the allocation-free solve on the caller's buffers) or "adjoint".
    grid: uniform cells (20 long in x), the reference's SML grid or the large
    workload's tanh-stretched one.  bc: "open" convective outflow and periodic
    z, "channel" zero-gradient outflow and slip walls, "cavity" the
    reference's lid-driven box.  mg: the V-cycle preconditioner; mixed: its
    cycle in FP32."""
    c = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "grid": "uniform", "bc": "open", "solver": "BICGSTAB", "op": "ELL",
         "mg": False, "mixed": False, "conv": "QUICK", "les": False, "tol": 1e-10, "maxit": 5000, "steps": 3}
    c.update(over)
    return c


def listed():
    return [
        # the grid of the parity tests and of the smoke check: launches and host latency
        _case("run", 32, 16, 8, name="run 32x16x8", bc="channel", steps=4),
        # the CPU-sized workload as configured: Jacobi BiCGSTAB to 1e-10 on 32768 rows
        _case("run", 128, 64, 4, name="run 128x64x4", steps=3),
        # the reference's compiled-in case: SML grid, lid-driven table, its default
        # matrix-free operator and its 1e-3 criterion
        _case("run", 190, 210, 40, name="run native 190x210x40", grid="native", bc="cavity", op="SPE", tol=1e-3, steps=4),
        # a ragged grid with the other options in use: linear upwind, Smagorinsky, slip walls in z
        _case("run", 150, 75, 27, name="run ragged LUD LES", bc="channel", op="ELL", conv="LUD", les=True, tol=1e-6,
              steps=3),
        # the reference's own SOR (P_SOLVER_SOR) in the step, at the reference's criterion
        _case("run", 96, 48, 24, name="run SorPipeLine", bc="channel", solver="SOR_PIPELINE", tol=1e-3, maxit=1500, steps=3),
        # production runs at 8.4M cells: every pass to 1e-10 with the multigrid preconditioner ...
        _case("run", 512, 256, 64, name="run 512x256x64 MG", op="SPE", mg=True, steps=3),
        # ... the same with the FP32 cycle ...
        _case("run", 512, 256, 64, name="run 512x256x64 MG mixed", op="SPE", mg=True, mixed=True, steps=3),
        # ... and the largest workload, 67M cells on stretched axes
        _case("run", 1024, 512, 128, name="run 1024x512x128 MG mixed", grid="stretched", mg=True, mixed=True, steps=2),
        # the reference's algorithm at 8.4M rows, Jacobi BiCGSTAB on the ELL operator,
        # bounded by its iteration cap (the full solve meets the cap of 5000)
        _case("poisson", 512, 256, 64, name="poisson 512x256x64 ELL", bc="channel", maxit=150),
        # one multigrid solve on extents that stop halving early
        _case("poisson", 200, 104, 40, name="poisson 200x104x40 MG", bc="channel", op="SPE", mg=True),
        # the solve on the caller's device arrays, for callers that may not allocate
        _case("device", 64, 32, 32, name="device 64x32x32"),
        # gradient of the mean drag: the adjoint workload's grid, a short objective window
        _case("adjoint", 256, 128, 32, name="adjoint 256x128x32", mg=True, steps=4),
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run small", "run mid", "run sor", "run mg", "poisson", "poisson mg", "device", "adjoint"])
    if kind == "run small":
        return _case("run", _between(rng, 16, 64), _between(rng, 8, 32), 2 * rng.randint(2, 8),
                     bc=rng.choice(["open", "channel"]), op=rng.choice(["ELL", "SPE"]), maxit=1000,
                     tol=rng.choice([1e-6, 1e-8, 1e-10]), steps=rng.randint(2, 4))
    if kind == "run mid":
        return _case("run", _between(rng, 64, 256), _between(rng, 32, 160), _between(rng, 4, 48), bc="channel",
                     op=rng.choice(["ELL", "SPE"]), conv=rng.choice(["QUICK", "LUD", "UD"]), les=rng.random() < 0.5,
                     tol=rng.choice([1e-3, 1e-6]), maxit=400, steps=rng.randint(2, 3))
    if kind == "run sor":
        return _case("run", _between(rng, 32, 160), _between(rng, 16, 80), _between(rng, 4, 40), bc="channel",
                     solver="SOR_PIPELINE", tol=1e-3, maxit=800, steps=2)
    if kind == "run mg":
        return _case("run", 32 * rng.randint(3, 16), 16 * rng.randint(3, 16), 8 * rng.randint(2, 8),
                     bc=rng.choice(["open", "channel"]), op=rng.choice(["SPE", "ELL"]), mg=True,
                     mixed=rng.random() < 0.5, steps=2)
    if kind == "poisson":
        return _case("poisson", _between(rng, 48, 512), _between(rng, 24, 256), _between(rng, 8, 64), bc="channel",
                     op=rng.choice(["ELL", "SPE"]), maxit=100)
    if kind == "poisson mg":
        return _case("poisson", 8 * rng.randint(4, 48), 8 * rng.randint(2, 24), 4 * rng.randint(2, 12), bc="channel",
                     op=rng.choice(["SPE", "ELL"]), mg=True)
    if kind == "device":
        return _case("device", _between(rng, 16, 160), _between(rng, 8, 80), _between(rng, 4, 40), tol=1e-8, maxit=2000)
    return _case("adjoint", 32 * rng.randint(2, 8), 16 * rng.randint(2, 8), 8 * rng.randint(1, 4), mg=True,
                 steps=rng.randint(2, 4))


# ---------------------------------------------------------------------------
# set-up
# ---------------------------------------------------------------------------

def _grid(case):
    n = (case["nx"], case["ny"], case["nz"])
    if case["grid"] == "native":
        return solver.native_grid()
    if case["grid"] == "stretched":
        return configs.cylinder_1024x512x128().grid
    h = 20.0 / n[0] if n[0] >= 64 else 0.25
    return solver.uniform_grid(n, tuple(h * m for m in n))


def _params(case, grid):
    if case["bc"] == "cavity":
        p = solver.default_params()
        p.source_index_quirk = 0
    else:
        if case["grid"] == "stretched":
            cx, cy, re, dt = 10.0, 10.0, 300.0, 2.5e-4
        else:
            cx, cy, re, dt = 0.25 * grid.lx, 0.5 * grid.ly, 100.0, 0.0128 * grid.lx / case["nx"]
        p = configs.cylinder_params(re, dt, cx, cy, 1.0, case["tol"])
        if case["bc"] == "open":
            configs.outflow_periodic_bc(p)
    p.tol, p.maxit = case["tol"], case["maxit"]
    p.solver, p.op = SOLVERS[case["solver"]], OPS[case["op"]]
    p.convection, p.les = CONV[case["conv"]], int(case["les"])
    if case["mg"]:
        p.precond = capi.CFD_PRECOND_MG
    if case["mixed"]:
        p.precision, p.mixed_mode = capi.CFD_MIXED, capi.CFD_MIXED_PC32
    return p


def _pinned(n):
    return torch.empty(n, dtype=torch.float64, pin_memory=torch.cuda.is_available())


def _rhs(case, seed):
    """The pressure right-hand side of a standalone solve: seeded N(0,1), zero mean."""
    g = torch.Generator().manual_seed(int(seed))
    b = torch.randn(case["nx"] * case["ny"] * case["nz"], dtype=torch.float64, generator=g)
    return b - b.mean()


def prepare(case, seed):
    grid = _grid(case)
    p = _params(case, grid)
    s = {"kind": case["kind"], "case": case, "seed": int(seed)}
    if case["kind"] == "device":
        # the caller's slot-major ELL operator, right-hand side, start value and solution on the device
        p.periodic_z = p.outflow_convective = 0
        with solver.Simulation(grid, p) as sim:
            sim.init_state()
            sim.createPressureMatrix()
            col, val = sim.ell()
        dev = torch.device("cuda", 0)
        s["col"], s["val"] = torch.from_numpy(col).to(dev), torch.from_numpy(val).to(dev)
        s["b"] = _rhs(case, seed).to(dev)
        s["x0"] = torch.zeros_like(s["b"])
        s["x"] = torch.empty_like(s["b"])
        return s
    sim = solver.Simulation(grid, p)
    s["sim"] = sim
    if case["kind"] != "poisson":
        s["out"] = {k: _pinned(sim.G) for k in ("u", "v", "w", "p")}
    if case["kind"] == "poisson":
        sim.init_state()
        sim.createPressureMatrix()
        if case["op"] == "SPE":
            sim.setupPressure()
        sim.upload(capi.RHS, _rhs(case, seed).numpy())
        s["x0"] = _pinned(sim.N).zero_()
        s["x"] = _pinned(sim.N)
    elif case["kind"] == "adjoint":
        sim.setup(noise=1e-3, seed=seed)
        s["u_in"] = adjoint.smoothed_inflow(case["ny"], seed=seed)
        s["problem"] = adjoint.DragProblem(sim, case["steps"], case["steps"] // 2, 2, noise=1e-3, seed=int(seed))
    else:
        sim.setup(noise=1e-3, seed=seed)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def _dptr(t):
    return C.cast(t.data_ptr(), C.POINTER(C.c_double))


def _fetch(sim, field, t):
    capi.check(sim.lib.cfd_download(sim.h, field, _dptr(t), t.numel()), "cfd_download")


def _fields(s):
    for k, f in (("u", capi.T0_U), ("v", capi.T0_V), ("w", capi.T0_W), ("p", capi.P)):
        _fetch(s["sim"], f, s["out"][k])
    return s["out"]


def run(s):
    case = s["case"]
    if s["kind"] == "device":
        s["x"].copy_(s["x0"])
        it, rel = C.c_int(), C.c_double()
        ptr = [C.c_void_p(s[k].data_ptr()) for k in ("col", "val", "b", "x")]
        stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        capi.check(capi.load().cfd_bicgstab_ell_noalloc(*ptr, s["b"].numel(), case["tol"], case["maxit"], stream,
                                                        C.byref(it), C.byref(rel)), "cfd_bicgstab_ell_noalloc")
        return {"x": s["x"]}
    sim = s["sim"]
    if s["kind"] == "poisson":
        capi.check(sim.lib.cfd_upload(sim.h, capi.X, _dptr(s["x0"]), sim.N), "cfd_upload")
        sim.solve()
        _fetch(sim, capi.X, s["x"])
        return {"x": s["x"]}
    if s["kind"] == "adjoint":
        J = s["problem"].run(s["u_in"], 1.001)
        g_uin, g_gain, _ = sim.adjoint_backward()
        return dict(_fields(s), J=J, g_uin=g_uin, g_gain=g_gain)
    sim.init_state(1e-3, s["seed"])
    for _ in range(case["steps"]):
        st = sim.step()
    return dict(_fields(s), cd=np.array(st.cd[:st.n_passes]), cl=np.array(st.cl[:st.n_passes]))


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    """Each step reads the velocity and the solid fraction and writes the
    velocity, the pressure and the force; each of its solves reads a
    right-hand side and writes a solution.  Operations: the predictor (about
    250 a cell) and one operator application and update per solve (30 a row);
    the iterations a solve takes beyond the first are not counted."""
    n = case["nx"] * case["ny"] * case["nz"]
    if case["kind"] == "device":  # the caller's matrix is an input here
        return {"bytes": 7 * n * 12.0 + 24.0 * n, "flops": 30.0 * n}
    if case["kind"] == "poisson":
        return {"bytes": 24.0 * n, "flops": 30.0 * n}
    solves = 4 * (case["steps"] - 1)
    step = {"bytes": (11.0 * case["steps"] + 2.0 * solves) * 8 * n, "flops": (250.0 * case["steps"] + 30.0 * solves) * n}
    if case["kind"] == "adjoint":  # the steps, the steps again, and their transposes
        return {k: 3.0 * v for k, v in step.items()}
    return step


# ---------------------------------------------------------------------------
# reference values in 64 bits
# ---------------------------------------------------------------------------

def _axis(n, h, dirichlet_hi):
    """-d2/dx2 on n uniform cells of width h: Neumann below, Neumann or p = 0
    in the first ghost cell above."""
    a = torch.zeros(n, n, dtype=torch.float64)
    i = torch.arange(n - 1)
    a[i, i + 1] = a[i + 1, i] = -1.0 / (h * h)
    d = torch.full((n,), 2.0 / (h * h), dtype=torch.float64)
    d[0] -= 1.0 / (h * h)
    if not dirichlet_hi:
        d[-1] -= 1.0 / (h * h)
    a[torch.arange(n), torch.arange(n)] = d
    return a


def exact(case, seed):
    """The solution of the walls' operator (p = 0 past the outflow face) by
    diagonalising each axis.  Timesteps and the adjoint end iterative solves
    at a tolerance and have no such value here, nor has a capped solve."""
    if case["kind"] not in ("poisson", "device") or (case["kind"] == "poisson" and not case["mg"]):
        return None
    n = (case["nx"], case["ny"], case["nz"])
    if n[0] * n[1] * n[2] > 1 << 24:
        return None
    h = 20.0 / n[0] if n[0] >= 64 else 0.25
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    axes = [_axis(m, h, q == 0) for q, m in enumerate(n)]
    eig = [torch.linalg.eigh(a) for a in axes]
    lam = [e[0].to(dev) for e in eig]
    vec = [e[1].to(dev) for e in eig]
    diag = [torch.diagonal(a).to(dev) for a in axes]
    d3 = diag[0][:, None, None] + diag[1][None, :, None] + diag[2][None, None, :]
    f = _rhs(case, seed).to(dev).reshape(n) * d3  # the solver's system is Jacobi-scaled: (1 / diag) L x = b

    def along(t, m, axis):
        return torch.tensordot(t.movedim(axis, -1).contiguous(), m, dims=1).movedim(-1, axis)

    for q in range(3):
        f = along(f, vec[q], q)
    f = f / (lam[0][:, None, None] + lam[1][None, :, None] + lam[2][None, None, :])
    for q in range(3):
        f = along(f, vec[q].T.contiguous(), q)
    return {"x": f.reshape(-1)}
