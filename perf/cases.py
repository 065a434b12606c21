"""Workloads of the SIMPLE solver that its speed is judged by.

Every case goes through the package's public entry points on one GPU.  Two
kinds of pass stand for what a user's program does:

* ``iterate``: a whole run from the initial state, a few SIMPLE iterations
  (all solves converged tightly), the cell fields copied back;
* ``momentum`` / ``pressure``: one phase of the SIMPLE loop on a resident
  case, as a host driver makes it: velocities set, momentum assembly and its
  three solves, velocities read back; or the pressure-correction solve of an
  assembled system and the correction read back.

The sizes run from a few thousand cells, where launches set the time, to
millions, where memory does; the meshes are uniform hexahedra (cavity),
jittered hexahedra with a tenth split into tetrahedra (channel), jittered
hexahedra (the turbulent channel) and jittered tetrahedra (the backward-facing
step), the solvers those that the benchmark's workloads and the package's
defaults name, in FP64 and in mixed precision.
"""
import numpy as np
import torch

import sysu_cfd_parallel_amd as s

# pressure-correction and momentum tolerances of the benchmark's workloads
RTOL = {"pressure": 1e-6, "momentum": 1e-8}
MAXIT = 20000


def listed():
    return [
        # a small laminar run: launches and host latency count
        {"name": "cavity16_run", "pass": "iterate", "mesh": "cavity", "n": 16, "solver": "gmres30_jacobi",
         "precision": "fp64", "steps": 2, "extra": "none"},
        # the laminar lid-driven cavity of the benchmark, a few of its iterations
        {"name": "cavity32_run", "pass": "iterate", "mesh": "cavity", "n": 32, "solver": "gmres30_jacobi",
         "precision": "fp64", "steps": 4, "extra": "none"},
        # an unsteady run with limited gradients and the energy equation
        {"name": "cavity24_unsteady", "pass": "iterate", "mesh": "cavity", "n": 24, "solver": "gmres30_jacobi",
         "precision": "fp64", "steps": 1, "extra": "unsteady"},
        # k-epsilon over tetrahedra with the package's default solvers
        # (GMRES and CG with ILU(0))
        {"name": "step4_keps_run", "pass": "iterate", "mesh": "step", "n": 4, "solver": "default",
         "precision": "fp64", "steps": 1, "extra": "keps"},
        # the momentum phase of the mixed-precision channel
        {"name": "channel100_momentum_mixed", "pass": "momentum", "mesh": "channel", "n": 100,
         "solver": "gmres50_jacobi", "precision": "mixed"},
        # the momentum phase on tetrahedra with the default solver
        {"name": "step6_momentum_ilu", "pass": "momentum", "mesh": "step", "n": 6, "solver": "default",
         "precision": "fp64"},
        # pressure solves of the channel: mixed at two sizes, the FP64 path
        {"name": "channel100_pressure_mixed", "pass": "pressure", "mesh": "channel", "n": 100,
         "solver": "gmres50_jacobi", "precision": "mixed"},
        {"name": "channel150_pressure_mixed", "pass": "pressure", "mesh": "channel", "n": 150,
         "solver": "gmres50_jacobi", "precision": "mixed"},
        {"name": "channel90_pressure_fp64", "pass": "pressure", "mesh": "channel", "n": 90,
         "solver": "gmres50_jacobi", "precision": "fp64"},
        # the default pressure solver, CG with ILU(0), on tetrahedra
        {"name": "step6_pressure_cg_ilu", "pass": "pressure", "mesh": "step", "n": 6, "solver": "default",
         "precision": "fp64"},
        # the turbulent channel's pressure solve, mixed GMRES with ILU(0)
        {"name": "hexchannel100_pressure_ilu_mixed", "pass": "pressure", "mesh": "hexchannel", "n": 100,
         "solver": "gmres50_ilu", "precision": "mixed"},
        # a parameter sweep: cavities of uneven sizes solved as one batch
        {"name": "sweep12_pressure_mixed", "pass": "pressure", "mesh": "sweep", "n": 12,
         "solver": "gmres30_jacobi", "precision": "mixed"},
    ]


# what draw() spreads its sizes over: (pass, mesh, solver, precision, extra, smallest n, largest n)
RANGES = [
    ("iterate", "cavity", "gmres30_jacobi", "fp64", "none", 9, 40),
    ("iterate", "cavity", "gmres30_jacobi", "fp64", "unsteady", 9, 28),
    ("iterate", "step", "default", "fp64", "keps", 2, 4),
    ("momentum", "channel", "gmres50_jacobi", "mixed", "", 24, 120),
    ("momentum", "channel", "gmres50_jacobi", "fp64", "", 24, 100),
    ("momentum", "step", "default", "fp64", "", 2, 6),
    ("pressure", "channel", "gmres50_jacobi", "mixed", "", 24, 150),
    ("pressure", "channel", "gmres50_jacobi", "fp64", "", 24, 110),
    ("pressure", "step", "default", "fp64", "", 2, 6),
    ("pressure", "hexchannel", "gmres50_ilu", "mixed", "", 24, 100),
    ("pressure", "sweep", "gmres30_jacobi", "mixed", "", 3, 12),
]


def draw(rng):
    what, mesh, solver, precision, extra, lo, hi = rng.choice(RANGES)
    n = round(lo * (hi / lo) ** rng.random())
    case = {"pass": what, "mesh": mesh, "n": n, "solver": solver, "precision": precision}
    if what == "iterate":
        case["steps"] = rng.randint(1, 3) if extra == "none" else 1
        case["extra"] = extra
    elif mesh != "sweep":
        # the channel's and the step's proportions vary too
        case["stretch"] = round(rng.uniform(0.6, 1.0), 3)
    return case


# ---- meshes and parameters

def _dims(case):
    """Cells of the channel's box: n along x, half of it across, about n in span."""
    n = case["n"]
    return n, max(3, n // 2), max(3, int(n * case.get("stretch", 1.0)) * (5 if case["mesh"] == "hexchannel" else 8) // 8)


def _sweep_edges(n):
    return [int(e) for e in np.random.default_rng(2024).integers(16, 65, size=n)]


def _build(case, re):
    """The mesh (the same for every seed) with the viscosity of the run's Reynolds number."""
    kind, n = case["mesh"], case["n"]
    if kind == "cavity":
        return s.cavity(n, re=re)
    if kind == "channel":
        return s.channel(*_dims(case), jitter=0.15, split=0.10, re=re)
    if kind == "hexchannel":
        return s.channel(*_dims(case), jitter=0.10, re=re)
    if kind == "step":
        return s.step(n, downstream=max(6.0, 30.0 * case.get("stretch", 1.0)), jitter=0.10, tets=True,
                      turbulent=case.get("extra") == "keps", re=re)
    return [s.cavity(e, re=re * (1 + 0.1 * k)) for k, e in enumerate(_sweep_edges(n))]


def _params(case):
    p = s.default_params()
    p.residual_steady = 0.0
    p.precision = s.MIXED if case["precision"] == "mixed" else s.FP64
    p.autotune = 1
    p.graphs = 0 if case["mesh"] == "channel" else 1
    name = case["solver"]
    if name != "default":
        restart, pc = int(name[5:7]), s.PC_ILU0 if name.endswith("ilu") else s.PC_JACOBI
        s.set_all_ksp(p, s.KSP_GMRES, restart, pc, maxit=MAXIT)
        if case["precision"] == "mixed" and pc == s.PC_JACOBI:
            p.inner_order = 2
    if case["pass"] == "iterate":
        # whole runs: every solve to a tight tolerance, so that the fields
        # depend on the equations and not on where the solver stopped
        for k in range(3):
            p.ksp[k].rtol, p.ksp[k].maxit = 1e-11, MAXIT
        if case["extra"] == "keps":
            p.turb_model = 1
            p.urf[3] = 0.3
        elif case["extra"] == "unsteady":
            p.steady, p.time_scheme, p.dt, p.total_time = 0, 2, 0.05, 1e6
            p.max_outer_step, p.limiter, p.solve_energy = 3, 1, 1
    return p


def _flow(xyz, rng, base):
    """A developing velocity and pressure: the bulk flow and a few smooth modes."""
    lo, hi = xyz.min(axis=0), xyz.max(axis=0)
    t = (xyz - lo) / (hi - lo)
    out = []
    for k in range(4):
        f = np.full(len(xyz), base if k == 0 else 0.0)
        if k == 0:
            f *= 4.0 * t[:, 1] * (1.0 - t[:, 1]) * 0.3 + 0.7
        for _ in range(3):
            wave = rng.integers(1, 4, size=3) * np.pi
            phase = rng.uniform(0, 2 * np.pi, size=3)
            f = f + 0.1 * np.prod(np.cos(t * wave + phase), axis=1)
        out.append(f)
    return out


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    base_re = {"cavity": 100.0, "sweep": 150.0, "step": 5000.0 if case.get("extra") == "keps" else 400.0}
    re = base_re.get(case["mesh"], 1000.0) * float(rng.uniform(0.9, 1.1))
    mesh = _build(case, re)
    solver = (s.BatchSolver if case["mesh"] == "sweep" else s.Solver)(mesh, _params(case))
    state = {"case": case, "solver": solver}
    if case["pass"] == "iterate":
        return state
    # a flow in mid-run: velocities and pressure, their fluxes, and for the
    # pressure solve the assembled system
    base = 0.0 if case["mesh"] in ("cavity", "sweep") else 1.0
    u, v, w, p = _flow(solver.dbls("CELL_X").reshape(-1, 3), rng, base)
    for name, f in (("U", u), ("V", v), ("W", w), ("P", 0.1 * p)):
        solver.set(name, f)
    solver.call("bc_velocity")
    solver.call("build_velocity_matrix")
    solver.call("cal_ru_face")
    if case["pass"] == "pressure":
        solver.call("bc_velocity")
        solver.call("build_pressure_matrix")
    else:
        state["velocity"] = (u, v, w)
    solver.call("synchronize")
    return state


def run(state):
    case, solver = state["case"], state["solver"]
    if case["pass"] == "iterate":
        solver.call("init_flow_field")
        _, steps = solver.iterate(case["steps"])
        names = ["U", "V", "W", "P"] + (["TE", "ED"] if case["extra"] == "keps" else []) \
            + (["T"] if case["extra"] == "unsteady" else [])
        return {"steps": steps, **{k: solver.get(k) for k in names}}
    if case["pass"] == "momentum":
        for name, f in zip("UVW", state["velocity"]):
            solver.set(name, f)
        solver.call("calculate_velocity", None)
        return {k: solver.get(k) for k in "UVW"}
    solver.solve_pressure(RTOL["pressure"], MAXIT)
    return solver.get("DELTAP")


def _cells(case):
    kind, n = case["mesh"], case["n"]
    if kind == "cavity":
        return n ** 3
    if kind == "sweep":
        return sum(e ** 3 for e in _sweep_edges(n))
    if kind == "step":
        length = max(6.0, 30.0 * case.get("stretch", 1.0))
        return int((4.0 + 2.0 * length) * 4.0 * 6 * n ** 3)
    nx, ny, nz = _dims(case)
    return nx * ny * nz * 3 // 2 if kind == "channel" else nx * ny * nz


def work(case):
    """Bytes and operations that a pass moves at least: each system's matrix
    (values, columns), right-hand side and solution once, and for the
    assembly the mesh and the fields.  An iterative solve reads them once per
    iteration; the count depends on the data and is left out."""
    n = _cells(case)
    nnz = n * (5 if case["mesh"] == "step" else 7)
    system = 12 * nnz + 16 * n
    assembly = n * (5 if case["mesh"] == "step" else 6) * 100 + 30 * 8 * n
    if case["pass"] == "pressure":
        return {"bytes": system, "flops": 2 * nnz}
    if case["pass"] == "momentum":
        return {"bytes": 12 * nnz + 3 * 24 * n + assembly, "flops": 6 * nnz + 300 * n}
    solves = 4 + (2 if case["extra"] == "keps" else 0) + (1 if case["extra"] == "unsteady" else 0)
    passes = case["steps"] * (2 if case["extra"] == "unsteady" else 1)
    return {"bytes": passes * (solves * system + 3 * assembly), "flops": passes * (2 * solves * nnz + 1000 * n)}


# ---- the exact solutions of the linear systems, in 64 bits with torch

def _csr(solver, field):
    dev = torch.device("cuda")
    ptr = torch.from_numpy(solver.ints("CSR_ROWPTR").astype(np.int64)).to(dev)
    col = torch.from_numpy(solver.ints("CSR_COL").astype(np.int64)).to(dev)
    val = torch.from_numpy(solver.get(field)).to(dev)
    row = torch.repeat_interleave(torch.arange(len(ptr) - 1, device=dev), ptr[1:] - ptr[:-1])
    return row, col, val, len(ptr) - 1


def _matvec(row, col, val, n):
    ptr = torch.zeros(n + 1, dtype=torch.int64, device=val.device)
    ptr[1:] = torch.cumsum(torch.bincount(row, minlength=n), 0)
    a = torch.sparse_csr_tensor(ptr, col, val, (n, n))
    return lambda x: (a @ x[:, None])[:, 0]


def _conjugate_gradients(mv, d, b, most):
    """Jacobi-preconditioned CG as far as 64 bits take it."""
    x, r = torch.zeros_like(b), b.clone()
    z = r / d
    p, rz = z.clone(), r @ z
    best, start, since = rz, rz, 0
    for k in range(most):
        q = mv(p)
        a = rz / (p @ q)
        x += a * p
        r -= a * q
        z = r / d
        new = r @ z
        p = z + (new / rz) * p
        rz = new
        if k % 50 == 49 and float(rz / start) < 1e-30:
            break
    return x


def _bicgstab(mv, d, b, most):
    """Jacobi-preconditioned BiCGStab as far as 64 bits take it."""
    x, r = torch.zeros_like(b), b / d
    r0, p = r.clone(), r.clone()
    rho, norm = r0 @ r, float(torch.linalg.vector_norm(r))
    for _ in range(most):
        v = mv(p) / d
        a = rho / (r0 @ v)
        h = r - a * v
        t = mv(h) / d
        w = (t @ h) / (t @ t)
        x += a * p + w * h
        r = h - w * t
        if float(torch.linalg.vector_norm(r)) < 1e-15 * norm:
            break
        new = r0 @ r
        p = r + (new / rho) * (a / w) * (p - w * v)
        rho = new
    return x


def _ilu_weights(row, col, val, n, d):
    """w = M^T 1 for M the ILU(0) product of a symmetric A with A 1 = 0 whose
    graph has no triangles (hexahedra; hexahedra cut into six tetrahedra): M
    differs from A by the dropped fill l_ij u_jk, and the factors keep A's
    off-diagonal entries over the pivots."""
    low = col < row
    i, j, a = row[low], col[low], val[low]
    u = d.clone()
    for _ in range(2000):  # exact after as many turns as the factorisation has levels
        new = d - torch.zeros_like(d).index_add_(0, i, a * a / u[j])
        same = bool(torch.all((new - u).abs() <= 1e-14 * d))
        u = new
        if same:
            break
    down = torch.zeros_like(d).index_add_(0, j, a)  # sum of a_ij over i > j
    return torch.zeros_like(d).index_add_(0, i, a / u[j] * (down[j] - a))


def exact(case, seed):
    if case["pass"] == "iterate":
        return None  # a whole nonlinear run has no short restatement
    state = prepare(case, seed)
    solver = state["solver"]
    if case["pass"] == "momentum":
        for name, f in zip("UVW", state["velocity"]):
            solver.set(name, f)
        solver.call("build_velocity_matrix")
    row, col, val, n = _csr(solver, "AU" if case["pass"] == "momentum" else "AP")
    mv = _matvec(row, col, val, n)
    d = torch.zeros(n, dtype=torch.float64, device=val.device).index_add_(0, row[row == col], val[row == col])
    rhs = lambda name: torch.from_numpy(solver.get(name)).to(val.device)  # noqa: E731
    if case["pass"] == "momentum":
        return {k: _bicgstab(mv, d, rhs("B%s_RHS" % k), 2000) for k in "UVW"}
    # the pressure correction is known up to a constant per case, which the
    # preconditioner fixes: M x stays in the range of A, whose rows sum to 0
    x = _conjugate_gradients(mv, d, rhs("BP_RHS"), 6000)
    weight = _ilu_weights(row, col, val, n, d) if case["solver"] in ("default", "gmres50_ilu") else d
    cuts = solver.layout["cell"].tolist() if case["mesh"] == "sweep" else [0, n]
    for a, e in zip(cuts[:-1], cuts[1:]):
        x[a:e] -= (weight[a:e] @ x[a:e]) / weight[a:e].sum()
    return x
