"""Timed workloads of the explicit residual path, the viscous terms, the BCSR
solvers, served batches and the mesh build, each through the package's public
entry points.

A case is a dict of plain values.  ``listed()`` gives the fixed cases,
``draw(rng)`` one more of the same ranges, ``prepare(case, seed)`` what a
program holds before the call (an uploaded mesh and its configuration, a
matrix handle, the initial states), ``run(state)`` one pass, ``work(case)``
the bytes and operations that the pass cannot do without and
``exact(case, seed)`` a 64-bit solution by plain torch where one exists.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from subfv_amd import lowmach
from subfv_amd import meshgen as mg
from subfv_amd.api import Bcsr, Solver, make_config
from subfv_amd.serve import Batch

ZERO = (0.0, 0.0, 0.0, 0.0, 0.0)


def _run_case(name, mesh, n, **kw):
    c = {"what": "run", "mesh": mesh, "n": n, "scheme": "multi_point", "order": 1, "method": 4, "time": "fe",
         "steps": 1, "viscous": "none", "arith": "exact", "state": "vortex"}
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one residual by the reference's compute_rhs_ns on a small 3-D mesh:
        # the smallest call a Fortran host makes, launches and latency only
        {"name": "residual_hex13", "what": "residual", "mesh": "hex", "n": 13, "scheme": "multi_point", "order": 2,
         "method": 4, "state": "vortex"},
        # the first-order parity workload: Sod on the jittered 128^2 quads for
        # 200 forward-Euler steps, a mesh too small to fill the GPU
        _run_case("sod_quad128_fe", "quad", 128, steps=200, state="sod"),
        # the plain explicit stage on a mesh that fills the GPU (1.2M prisms)
        _run_case("euler_tri768_fe", "tri", 768, steps=24),
        # the benchmark's default workload: 2.1M prisms, second order, viscous
        # (mu = 1e-3, Pr = 0.72), SSP-RK3
        _run_case("ns_tri1024_rk3", "tri", 1024, order=2, time="rk3", steps=3, viscous="constant"),
        # the same scheme with Sutherland's viscosity, whose nodal systems are
        # formed anew for every residual (odd grid size)
        _run_case("ns_tri255_sutherland", "tri", 255, order=2, time="rk3", steps=1, viscous="sutherland"),
        # the 3-D blast on tetrahedra with the reference's two-stage scheme
        _run_case("blast_tet40_two_stage", "tet", 40, order=2, steps=8, state="blast"),
        # viscous terms on tetrahedra: vertices of up to 36 sub-faces
        _run_case("ns_tet15_rk3", "tet", 15, order=2, time="rk3", steps=4, viscous="constant"),
        # second-order Euler with the fast arithmetic of the node sweep
        _run_case("euler_tri511_fast", "tri", 511, order=2, time="rk3", steps=4, arith="fast"),
        # the implicit low-Mach system, GMRES(30) to 1e-10, in FP64 ...
        {"name": "lowmach512_gmres", "what": "gmres", "n": 512, "precision": 0},
        # ... and with FP32 products inside FP64 restarts (odd size)
        {"name": "lowmach301_gmres_fp32", "what": "gmres", "n": 301, "precision": 1},
        # served solves: 40 resident instances of uneven sizes advanced together
        # by replayed graphs, each from a new two-state initial condition
        {"name": "batch40_fe", "what": "batch", "count": 40, "nmin": 16, "nmax": 120, "steps": 60},
        # build_mesh + geometry for a mesh that just arrived, on the device
        {"name": "mesh_build_tri200", "what": "mesh", "mesh": "tri", "n": 200},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["run", "run", "run", "viscous", "viscous", "residual", "gmres", "batch", "mesh"])
    if what == "residual":
        mesh = rng.choice(["hex", "tet", "quad", "tri"])
        n = _log_int(rng, 4, 20) if mesh in ("hex", "tet") else _log_int(rng, 8, 150)
        return {"what": "residual", "mesh": mesh, "n": n, "order": rng.choice([1, 2]),
                "scheme": rng.choice(["multi_point", "multi_point", "three_wave", "two_wave", "multi_point_pressure"]),
                "method": rng.choice([0, 2, 3, 4, 5, 6]), "state": "vortex"}
    if what == "gmres":
        return {"what": "gmres", "n": _log_int(rng, 48, 500), "precision": rng.choice([0, 1])}
    if what == "batch":
        return {"what": "batch", "count": rng.randint(3, 40), "nmin": 16, "nmax": rng.randint(40, 120),
                "steps": rng.choice([30, 45, 60])}
    if what == "mesh":
        mesh = rng.choice(["tri", "quad", "tet"])
        return {"what": "mesh", "mesh": mesh, "n": _log_int(rng, 8, 16) if mesh == "tet" else _log_int(rng, 40, 200)}
    if what == "viscous":
        mesh, law = rng.choice([("tri", "constant"), ("tri", "constant"), ("tri", "sutherland"), ("quad", "constant"),
                                ("quad", "sutherland"), ("tet", "constant"), ("hex", "constant")])
        top = {"tri": 400, "quad": 500, "tet": 15, "hex": 36}[mesh] if law == "constant" else 250
        return _run_case("", mesh, _log_int(rng, 6 if mesh in ("tet", "hex") else 24, top),
                         order=rng.choice([1, 2, 2]), time="rk3", steps=1 if law == "sutherland" else rng.randint(1, 6),
                         viscous=law)
    mesh = rng.choice(["quad", "tri", "tri", "tet", "hex"])
    n = {"quad": _log_int(rng, 24, 800), "tri": _log_int(rng, 24, 700), "tet": _log_int(rng, 6, 40),
         "hex": _log_int(rng, 6, 64)}[mesh]
    order = rng.choice([1, 1, 2])
    return _run_case("", mesh, n, order=order, method=rng.choice([2, 4, 4, 5]), time=rng.choice(["fe", "rk3"]),
                     scheme=rng.choice(["multi_point", "multi_point", "multi_point", "multi_point_iso", "three_wave",
                                        "modified_three_wave"]),
                     steps=rng.randint(3, 16), arith=rng.choice(["exact", "exact", "fast"]),
                     state=rng.choice(["sod", "vortex"]))


# --------------------------------------------------------------- preparation
def _mesh(kind, n, seed):
    make = {"quad": mg.quad_mesh, "tri": mg.tri_mesh, "tet": mg.tet_mesh, "hex": mg.hex_mesh}[kind]
    return make(n, seed=seed)


def _state(case, solver, seed):
    x = solver.elem_coord
    u = mg.uniform(seed, 40, np.arange(8, dtype=np.uint64))
    if case["state"] == "sod":
        return mg.init_1drp(x, 0.45 + 0.1 * u[0], [1.0, 0.1 * u[1], 0, 0, 1.0], [0.125, 0, 0, 0, 0.1])
    if case["state"] == "blast":
        return mg.blast_state(x, solver.elem_volume, 1.0 / case["n"], seed=seed)
    return mg.vortex_state(x, seed=seed, n_vortex=8)


def _solver(case, seed):
    s = Solver(0)
    mesh = _mesh(case["mesh"], case["n"], seed)
    s.build_mesh(mesh)
    s.set_config(make_config(case["scheme"], boundary_2d=mesh.boundary_2d, second_order=case["order"] == 2,
                             method=case["method"], cfl=0.4))
    viscous = case.get("viscous", "none")
    if viscous != "none":
        # untagged walls (zero viscous flux); the vortex state has T of about 3.5e-3
        s.set_diffusion(True, mu=1e-3, cv=720.19471, prandtl=0.72)
        if viscous == "sutherland":
            s.set_sutherland(True, mu0=1e-3, T0=3.5e-3)
    if case.get("arith") == "fast":
        s.set_arith(True)
    return s


def prepare(case, seed):
    what = case["what"]
    if what == "gmres":
        sysm = lowmach.build_system(case["n"], seed=seed)
        s = Solver(0)
        A = Bcsr(s, sysm["m"], sysm["b"], sysm["row"], sysm["col"], sysm["v"])
        return {"what": what, "solver": s, "A": A, "rhs": sysm["rhs"], "precision": case["precision"],
                "tol": 1e-10 * float(np.linalg.norm(sysm["rhs"]))}
    if what == "mesh":
        return {"what": what, "solver": Solver(0), "mesh": _mesh(case["mesh"], case["n"], seed)}
    if what == "batch":
        # the sizes belong to the case, the node jitter and the states to the seed
        k = np.arange(case["count"], dtype=np.uint64)
        u = [mg.uniform(case["count"] if j < 2 else seed, 60 + j, k) for j in range(8)]
        solvers, init = [], []
        for i in range(case["count"]):
            n = int(round(math.exp(math.log(case["nmin"]) + u[0][i] * math.log(case["nmax"] / case["nmin"]))))
            mesh = _mesh("quad" if u[1][i] < 0.5 else "tri", n, seed + i)
            s = Solver(0)
            s.build_mesh(mesh)
            s.set_config(make_config("multi_point", boundary_2d=True, cfl=0.4))
            solvers.append(s)
            init.append((0.3 + 0.4 * u[2][i], [0.1 + 0.9 * u[3][i], u[4][i] - 0.5, 0.0, 0.0, 0.1 + 0.9 * u[5][i]],
                         [0.1 + 0.9 * u[6][i], 0.0, 0.3 * u[4][i], 0.0, 0.1 + 0.9 * u[7][i]]))
        return {"what": what, "solvers": solvers, "init": init, "batch": Batch(0), "steps": case["steps"]}
    s = _solver(case, seed)
    st = {"what": what, "solver": s, "sol": _state(case, s, seed)}
    if what == "run":
        st["steps"] = case["steps"]
        st["time"] = 1 if case["time"] == "rk3" else 0
    return st


# ----------------------------------------------------------------- one pass
def run(state):
    what = state["what"]
    if what == "gmres":
        x, conv, _ = state["A"].gmres_diag(state["rhs"], state["tol"], 30, state["precision"])
        return {"x": x, "converged": int(conv)}
    if what == "mesh":
        s = state["solver"]
        s.build_mesh(state["mesh"])
        return {"elem_nto": s.mesh_i("elem_nto"), "left": s.mesh_i("sub_face_left_elem"),
                "right": s.mesh_i("sub_face_right_elem"), "area": s.mesh_d("sub_face_area"),
                "volume": s.elem_volume}
    if what == "batch":
        for s, (x, wl, wr) in zip(state["solvers"], state["init"]):
            s.init_1drp(x, wl, wr)
            s.set_time(0.0)
        state["batch"].run(state["solvers"], state["steps"], 1)
        state["batch"].wait()
        return [s.get_sol() for s in state["solvers"]]
    s = state["solver"]
    s.put_sol(state["sol"])
    if what == "residual":
        rhs, sl = s.compute_rhs_ns()
        return {"rhs": rhs, "sum_lambda": sl}
    s.set_time(0.0)
    t, dt = s.run(state["steps"], state["time"])
    return {"sol": s.get_sol(), "t": t, "dt": dt}


# ------------------------------------------------------ what a pass must do
def _counts(kind, n):
    """cells, vertices, sub-faces and sub-elements of the generated meshes"""
    if kind == "quad":
        return n * n, 2 * (n + 1) ** 2, 16 * n * n + 8 * n, 8 * n * n
    if kind == "tri":
        return 2 * n * n, 2 * (n + 1) ** 2, 24 * n * n + 8 * n, 12 * n * n
    if kind == "hex":
        return n ** 3, (n + 1) ** 3, 12 * n * n * (n + 1), 8 * n ** 3
    return 6 * n ** 3, (n + 1) ** 3, 36 * n ** 3 + 18 * n * n, 24 * n ** 3


def _stage(kind, n, order, viscous, update=True):
    """One residual (and update): the state in and out, the cell volumes, each
    sub-face's normal, area and two cells, the slots' cells and the vertex
    offsets; centroids and vertex coordinates in second order, sub-element
    volumes for the viscous terms.  Operations: the four nodal-solver
    iterations and the flux per sub-face, the 3x3 solves per vertex; the
    gradients and limiters; the viscous nodal systems."""
    C, V, SF, SE = _counts(kind, n)
    b = C * (88 if update else 96) + SF * 40 + SE * 4 + V * 4
    f = SF * 500 + V * 400 + C * 40
    if order == 2:
        b += C * 24 + V * 24
        f += SF * 600 + V * 400 + C * 500
    if viscous != "none":
        b += SE * 8
        f += V * 2500 if viscous == "constant" else V * 20000
    return b, f


def work(case):
    what = case["what"]
    if what == "gmres":
        m = case["n"] ** 2
        word = 8 if case["precision"] == 0 else 4
        # about 150 Arnoldi steps: the blocks, their columns, and x and y of the
        # product, and the basis built so far (15 columns on average) once
        per = 5 * m * (16 * word + 4) + 2 * 4 * m * 8 + 15 * 4 * m * word
        return {"bytes": 150 * per, "flops": 150 * (5 * m * 32 + 15 * 4 * m * 4)}
    if what == "mesh":
        C, V, SF, SE = _counts(case["mesh"], case["n"])
        return {"bytes": V * 24 + SE * 4 + C * 12 + SF * 16, "flops": SF * 60}
    if what == "batch":
        # sizes log-uniform in [nmin, nmax], half of them quads, half prisms
        a, b = math.log(case["nmin"]), math.log(case["nmax"])
        n2 = (math.exp(2 * b) - math.exp(2 * a)) / (2 * (b - a)) if b > a else math.exp(2 * a)
        n = int(math.sqrt(n2))
        q, t = _stage("quad", n, 1, "none"), _stage("tri", n, 1, "none")
        k = case["count"] * case["steps"] / 2
        return {"bytes": int(k * (q[0] + t[0])), "flops": int(k * (q[1] + t[1]))}
    if what == "residual":
        b, f = _stage(case["mesh"], case["n"], case["order"], "none", update=False)
        return {"bytes": b, "flops": f}
    b, f = _stage(case["mesh"], case["n"], case["order"], case["viscous"])
    stages = case["steps"] * (3 if case["time"] == "rk3" else (2 if case["order"] == 2 else 1))
    return {"bytes": stages * b, "flops": stages * f}


# ------------------------------------------------------------ 64-bit answers
def _block_solve(sysm):
    """J x = rhs by BiCGStab with block-Jacobi in torch FP64 on the GPU,
    restarted from the true residual until it stops falling."""
    m, b = sysm["m"], sysm["b"]
    dev = "cuda"
    k = sysm["col"].size // m  # every row of this system has the same number of blocks
    col = torch.from_numpy(sysm["col"].astype(np.int64) - 1).to(dev)
    v = torch.from_numpy(sysm["v"]).to(dev).reshape(m * k, b, b)  # [entry][column][row]
    rows = torch.arange(m, device=dev).repeat_interleave(k)
    Dinv = torch.linalg.inv(v[rows == col].transpose(1, 2).contiguous())
    rhs = torch.from_numpy(sysm["rhs"]).to(dev).reshape(m, b)

    def mul(x):
        return (v * x[col][:, :, None]).sum(1).reshape(m, k, b).sum(1)

    def prec(x):
        return (Dinv * x[:, None, :]).sum(2)

    def dot(x, y):
        return float((x * y).sum())

    x = torch.zeros_like(rhs)
    best, best_x = math.inf, x
    for _ in range(6):
        r = rhs - mul(x)
        n0 = math.sqrt(dot(r, r))
        if n0 >= 0.5 * best:
            break
        best, best_x = n0, x.clone()
        r0, p, rho = r.clone(), r.clone(), dot(r, r)
        for _ in range(600):
            ph = prec(p)
            q = mul(ph)
            alpha = rho / dot(r0, q)
            s = r - alpha * q
            sh = prec(s)
            t = mul(sh)
            om = dot(t, s) / dot(t, t)
            x = x + alpha * ph + om * sh
            r = s - om * t
            if math.sqrt(dot(r, r)) < 1e-8 * n0 or not math.isfinite(om):
                break
            new = dot(r0, r)
            p = r + (new / rho) * (alpha / om) * (p - om * q)
            rho = new
    return best_x.reshape(-1).cpu().numpy()


def exact(case, seed):
    """The solution of the linear systems.  The explicit runs are whole time
    loops of a nodal solver over a renumbered mesh, and the mesh build returns
    that numbering: neither has a short 64-bit form in plain numpy."""
    if case["what"] != "gmres":
        return None
    return {"x": _block_solve(lowmach.build_system(case["n"], seed=seed)), "converged": None}
