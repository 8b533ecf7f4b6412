"""Viscous terms on the device (diffusion.hip) against the oracle
(om_diffusion.c).  The device keeps the inverses of the nodal systems and
adds each cell's terms as one sum per vertex, where the reference multiplies
dense matrices and adds the terms one by one; results agree to round-off, not bit for bit: the residual within
1e-12 of the viscous terms' scale (measured: 2e-14 on tri 8^2, 4e-17 for the
point-implicit diagonal) and the state after 100 viscous steps within 1e-12
relative (measured: 1e-15 on tri, quad, 3-D hex and a 10-sub-element fan).
Tetrahedral meshes (36 sub-faces and 24 sub-elements at an interior vertex)
take the large-class kernels: inverses formed by a workgroup per vertex and
read from HBM."""
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle as O
from subfv_amd import meshgen as mg
from subfv_amd.api import Solver, SubfvError, make_config

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def solver():
    s = Solver(0)
    yield s
    s.close()


def smooth_state(xc, seed=5):
    rng = np.random.default_rng(seed)
    x, y, z = xc[:, 0], xc[:, 1], xc[:, 2]
    w = np.stack([1.0 + 0.2 * np.sin(3 * x + 1) * np.cos(2 * y) + 0.02 * rng.random(x.size),
                  0.3 * np.sin(2 * y + 0.5), -0.2 * np.cos(3 * x), 0.05 * np.sin(4 * z + x),
                  1.0 + 0.3 * np.cos(2 * x + y) + 0.02 * rng.random(x.size)], 1)
    return mg.primit_to_conserv(w)


CASES = {
    "quad9": (lambda: mg.quad_mesh(9), dict(), dict()),
    "tri7": (lambda: mg.tri_mesh(7), dict(), dict()),
    "quad8lr_dirichlet": (lambda: mg.quad_mesh(8, tags="lr"),
                          dict(bcs=[("freestream", (1.0, 0.2, 0.0, 0.0, 1.0)), ("outflowsupersonic", (0, 0, 0, 0, 0))]),
                          dict(bcs_v=[("dirichlet", (0.1, -0.05, 0.0)), ("neumann", (0, 0, 0))],
                               bcs_t=[("dirichlet", 1.5e-3), ("neumann", 0.0)])),
    "tet3": (lambda: mg.tet_mesh(3), dict(boundary_2d=False), dict()),  # large size class
}


@pytest.mark.parametrize("second", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_rhs_and_diag_match_oracle(solver, name, second):
    print(f"[gpu] diffusion rhs {name} second={second}", flush=True)
    mk, cfgkw, dkw = CASES[name]
    mesh = mk()
    solver.build_mesh(mesh)
    om = O.OracleMesh(mesh)
    sol = smooth_state(om.elem_coord)
    mu = 2e-3
    solver.set_config(make_config("multi_point", second_order=second, method=4, **cfgkw))
    solver.set_diffusion(True, mu=mu, **dkw)
    solver.put_sol(sol)
    solver.compute_rhs_ns()
    rhs = solver.get("rhs")
    diag = solver.get("diag")
    ocfg = O.make_config("multi_point", second_order=second, method=4, diffusion=True, mu=mu, **cfgkw, **dkw)
    r0, sl = om.compute_euler_flux(ocfg, sol)
    if second:
        g = om.compute_cell_grad(sol, 4)[0]
        r2, _ = om.compute_euler_flux(ocfg, sol, grad=g, second_order=True)
        r0 = om.flux_limiting(sol, r0, r2, sl, ocfg.cfl)
    rd, dd = om.add_diffusion(ocfg, sol)
    ref_rhs = r0 + rd
    scale_r = np.abs(rd).max(axis=0) + 1e-300
    scale_d = np.abs(dd).max()
    # Euler part bit-exact; the viscous part to 1e-12 of its scale
    assert np.all(np.abs(rhs - ref_rhs) <= 1e-12 * scale_r[None, :] + 1e-14 * np.abs(ref_rhs)), \
        np.abs(rhs - ref_rhs).max(axis=0) / scale_r
    assert np.abs(diag - dd).max() <= 1e-12 * scale_d
    solver.set_diffusion(False)


@pytest.mark.parametrize("scheme,second,ts", [("multi_point", False, 0), ("multi_point", True, 0),
                                              ("two_wave", True, 1)])
def test_viscous_time_loop_matches_oracle(solver, scheme, second, ts):
    print(f"[gpu] diffusion run {scheme} second={second} ts={ts}", flush=True)
    mesh = mg.tri_mesh(8)
    solver.build_mesh(mesh)
    om = O.OracleMesh(mesh)
    sol = smooth_state(om.elem_coord, 9)
    mu = 5e-3
    solver.set_config(make_config(scheme, second_order=second, method=4, cfl=0.3))
    solver.set_diffusion(True, mu=mu)
    solver.set_time(0.0)
    solver.put_sol(sol)
    solver.run(10, ts)
    got = solver.get_sol()
    st, ref, info = om.run(O.make_config(scheme, second_order=second, method=4, cfl=0.3, diffusion=True, mu=mu),
                           sol, 10, ts)
    assert st == 0
    rel = np.abs(got - ref).max() / np.abs(ref).max()
    assert rel <= 1e-12, rel
    solver.set_diffusion(False)


def fan_prism_mesh(k=5, layers=2):
    """k prisms around a vertical axis, extruded in `layers` layers: the axis
    vertices between layers have 2k sub-elements and 3k sub-faces (10 and
    15 for k = 5), more than the viscous apply stages in LDS."""
    ang = 2 * np.pi * np.arange(k) / k + 0.1
    pts = np.concatenate([[[0.0, 0.0]], np.stack([np.cos(ang), np.sin(ang)], 1)])
    coord = np.concatenate([np.column_stack([pts, np.full(len(pts), 0.4 * z)]) for z in range(layers + 1)])
    ev = []
    for lay in range(layers):
        o, o2 = lay * len(pts), (lay + 1) * len(pts)
        for q in range(k):
            a, b, c = 0, 1 + q, 1 + (q + 1) % k
            ev.append([o + a, o + b, o + c, o2 + a, o2 + b, o2 + c])
    ev = np.array(ev) + 1
    return mg.Mesh(coord, np.full(len(ev), 6, np.int32), ev.astype(np.int32).ravel(), boundary_2d=False, name="fan")


LONG_CASES = {
    "tri8": lambda: mg.tri_mesh(8),
    "hex3": lambda: mg.hex_mesh(3),  # 3-D interior vertices: 12 sub-faces, 8 sub-elements
    "fan5": fan_prism_mesh,          # 10 sub-elements: slot terms read from HBM
    "tet3": lambda: mg.tet_mesh(3),  # 36 sub-faces, 24 sub-elements: the large size class
}


@pytest.mark.parametrize("ts", [0, 1])
@pytest.mark.parametrize("name", list(LONG_CASES))
def test_viscous_100_steps_within_1e12(solver, name, ts):
    """100 second-order viscous steps (the reference's two-stage loop and
    SSP-RK3): the conserved states stay within 1e-12 relative of the
    oracle's, on a prism mesh, a 3-D hex mesh and a mesh whose vertices
    exceed the LDS staging of the viscous apply."""
    print(f"[gpu] viscous 100 steps {name} ts={ts}", flush=True)
    mesh = LONG_CASES[name]()
    solver.build_mesh(mesh)
    om = O.OracleMesh(mesh)
    sol = smooth_state(om.elem_coord, 9)
    kw = dict(boundary_2d=mesh.boundary_2d, second_order=True, method=4, cfl=0.3)
    solver.set_config(make_config("multi_point", **kw))
    solver.set_diffusion(True, mu=5e-3)
    solver.set_time(0.0)
    solver.put_sol(sol)
    solver.run(100, ts)
    got = solver.get_sol()
    solver.set_diffusion(False)
    st, ref, info = om.run(O.make_config("multi_point", diffusion=True, mu=5e-3, **kw), sol, 100, ts)
    assert st == 0
    rel = np.abs(got - ref).max() / np.abs(ref).max()
    assert rel <= 1e-12, rel


# (k, layers): the axis vertex between two layers has 2k sub-elements and 3k
# faces, all with unknowns of their own; with one layer k sub-elements, k such
# faces and k derived wall faces.  Edges of the size classes: 10 | 11 (32 or 64
# lanes per vertex), 21 | 22 and 24 (inverses in HBM), 37 | 39 (larger tiles),
# 63 (the most a byte code holds is 64).
@pytest.mark.parametrize("law", ["constant", "sutherland"])
@pytest.mark.parametrize("k,layers", [(3, 1), (10, 1), (11, 1), (7, 2), (22, 1), (8, 2), (13, 2), (21, 2)])
def test_vertex_size_classes_match_oracle(solver, k, layers, law):
    print(f"[gpu] viscous class fan k={k} layers={layers} {law}", flush=True)
    viscous_matches_oracle(solver, fan_prism_mesh(k, layers), law, dict(boundary_2d=False), {})


_FACES = {4: ([0, 1, 2], [0, 1, 3], [1, 2, 3], [0, 2, 3]),
          5: ([0, 1, 2, 3], [4, 5, 6, 7], [0, 1, 5, 4], [1, 2, 6, 5], [2, 3, 7, 6], [3, 0, 4, 7]),
          6: ([0, 1, 2], [3, 4, 5], [0, 1, 4, 3], [1, 2, 5, 4], [2, 0, 3, 5])}


def tag_boundary(mesh, tag):
    """The mesh with its boundary faces tagged: tag(centre) is 0 (untagged, the
    default wall) or a BC index."""
    off = mg.elem_offsets(mesh.kind)
    seen = {}
    for e, kind in enumerate(mesh.kind):
        v = mesh.elem_vert[off[e]:off[e + 1]]
        for f in _FACES[int(kind)]:
            seen.setdefault(frozenset(v[f].tolist()), []).append(v[f])
    nv, verts, tags = [], [], []
    for f in seen.values():
        t = tag(mesh.coord[f[0] - 1].mean(axis=0)) if len(f) == 1 else 0
        if t:
            nv.append(len(f[0]))
            verts.append(f[0])
            tags.append(t)
    mesh.bf_nvert, mesh.bf_tag = np.array(nv, np.int32), np.array(tags, np.int32)
    mesh.bf_vert = np.concatenate(verts).astype(np.int32)
    return mesh


def shell_mesh(k, rings):
    """One layer of a spherical shell: k prisms around each pole, k hexahedra
    in each of the rings - 1 belts between.  The numbering starts at one pole,
    so the other, with its k sub-elements, is the last vertex."""
    th = np.pi * (1 + np.arange(rings)) / (rings + 1)
    ph = 2 * np.pi * np.arange(k) / k
    ring = np.stack([np.outer(np.sin(th), np.cos(ph)), np.outer(np.sin(th), np.sin(ph)),
                     np.outer(np.cos(th), np.ones(k))], -1).reshape(-1, 3)
    pts = np.concatenate([[[0, 0, 1.0]], ring, [[0, 0, -1.0]]])
    n, south = len(pts), len(pts) - 1
    at = lambda r, q: 1 + r * k + q % k
    ev, kind = [], []
    for q in range(k):
        for low in ([0, at(0, q), at(0, q + 1)], [south, at(rings - 1, q + 1), at(rings - 1, q)]):
            ev.append(low + [v + n for v in low])
            kind.append(6)
        for r in range(rings - 1):
            low = [at(r, q), at(r + 1, q), at(r + 1, q + 1), at(r, q + 1)]
            ev.append(low + [v + n for v in low])
            kind.append(5)
    flat = np.concatenate([np.array(e) for e in ev]) + 1
    return mg.Mesh(np.concatenate([pts, 1.3 * pts]), np.array(kind, np.int32), flat.astype(np.int32),
                   boundary_2d=False, name="shell")


TAGGED = (dict(boundary_2d=False, bcs=[("freestream", (1.0, 0.2, 0.0, 0.0, 1.0)), ("outflowsupersonic", (0,) * 5)]),
          dict(bcs_v=[("dirichlet", (0.1, -0.05, 0.02)), ("neumann", (0, 0, 0))],
               bcs_t=[("dirichlet", 1.5e-3), ("dirichlet", 1.2e-3)]))


def viscous_matches_oracle(solver, mesh, law, cfgkw, dkw, sol=None, tol=1e-12):
    """rhs and diag of one first-order residual within 1e-12 of the viscous
    terms' scale, as for the meshes above."""
    solver.build_mesh(mesh)
    om = O.OracleMesh(mesh)
    suth = law == "sutherland"
    if sol is None:
        sol = warm_state(om.elem_coord) if suth else smooth_state(om.elem_coord)
    solver.set_config(make_config("multi_point", second_order=False, **cfgkw))
    solver.set_diffusion(True, mu=2e-3, **dkw)
    solver.set_sutherland(suth)
    try:
        solver.put_sol(sol)
        solver.compute_rhs_ns()
        rhs, diag = solver.get("rhs"), solver.get("diag")
    finally:
        solver.set_sutherland(False)
        solver.set_diffusion(False)
    ocfg = O.make_config("multi_point", second_order=False, diffusion=True, mu=2e-3, sutherland=suth, **cfgkw, **dkw)
    r0, _ = om.compute_euler_flux(ocfg, sol)
    rd, dd = om.add_diffusion(ocfg, sol)
    scale = np.abs(rd).max(axis=0) + 1e-300
    assert np.all(np.abs(rhs - (r0 + rd)) <= tol * scale[None, :] + 1e-14 * np.abs(r0 + rd)), \
        np.abs(rhs - r0 - rd).max(axis=0) / scale
    assert np.abs(diag - dd).max() <= tol * np.abs(dd).max()


@pytest.mark.parametrize("law", ["constant", "sutherland"])
@pytest.mark.parametrize("k,rings", [(8, 2), (10, 4), (13, 3)])
def test_largest_vertex_last_matches_oracle(solver, k, rings, law):
    """A tagged pole as the last vertex, larger than those before it: the
    wavefronts that round the launch up to whole workgroups lie past it."""
    print(f"[gpu] viscous shell k={k} rings={rings} {law}", flush=True)
    mesh = tag_boundary(shell_mesh(k, rings), lambda x: 1 if x[2] < -0.8 and x[0] > 0.0 and abs(x[1]) < 0.3 else 0)
    n_faces = O.OracleMesh(mesh).geti("vert_n_sub_faces")
    assert n_faces[-1] == n_faces.max() and -(-n_faces.size // 16) * 4 > -(-n_faces.size // 4)
    viscous_matches_oracle(solver, mesh, law, *TAGGED)


def mixed_tags(x):
    """untagged, Dirichlet and Neumann velocities (both with Dirichlet
    temperatures) in turn over the boundary"""
    return int(np.floor(7.3 * x[0] + 5.1 * x[1] + 3.7 * x[2])) % 3


# tagged vertices outside the 32-lane class: 64 lanes (hexahedra; a fan between
# two layers, with 11 and more stored faces) and a workgroup per vertex (tets)
@pytest.mark.parametrize("law", ["constant", "sutherland"])
@pytest.mark.parametrize("mk", [lambda: mg.hex_mesh(3), lambda: fan_prism_mesh(7, 2), lambda: fan_prism_mesh(12, 1),
                                lambda: mg.tet_mesh(3), lambda: fan_prism_mesh(16, 2)],
                         ids=["hex3", "fan7x2", "fan12", "tet3", "fan16x2"])
def test_tagged_boundaries_of_each_class_match_oracle(solver, mk, law):
    mesh = tag_boundary(mk(), mixed_tags)
    print(f"[gpu] viscous tagged {mesh.name} {mesh.n_elems} {law}", flush=True)
    assert set(np.unique(mesh.bf_tag)) == {1, 2}
    viscous_matches_oracle(solver, mesh, law, *TAGGED)


def pyramid_mesh(n, seed=3):
    """n^3 hexahedra, each split into six pyramids about a displaced centre:
    four sub-faces of a cell meet at its apex."""
    h = mg.hex_mesh(n)
    v = h.elem_vert.reshape(-1, 8)
    rng = np.random.default_rng(seed)
    centre = h.coord[v - 1].mean(axis=1) + 0.05 / n * rng.uniform(-1, 1, (len(v), 3))
    ids = h.n_vert + 1 + np.arange(len(v))
    faces = ([0, 1, 2, 3], [4, 7, 6, 5], [0, 4, 5, 1], [1, 5, 6, 2], [2, 6, 7, 3], [3, 7, 4, 0])
    ev = np.concatenate([np.column_stack([v[:, f], ids]) for f in faces])
    return mg.Mesh(np.concatenate([h.coord, centre]), np.full(len(ev), 7, np.int32), ev.astype(np.int32).ravel(),
                   boundary_2d=False, name="pyramid")


# the 64-lane class (12 stored faces at the apex) and the large one (36 faces at
# an inner corner)
@pytest.mark.parametrize("law", ["constant", "sutherland"])
@pytest.mark.parametrize("n", [1, 2])
def test_pyramids_match_oracle(solver, n, law):
    print(f"[gpu] viscous pyramids {n} {law}", flush=True)
    viscous_matches_oracle(solver, pyramid_mesh(n), law, dict(boundary_2d=False), {})


@pytest.mark.parametrize("law", ["constant", "sutherland"])
def test_viscous_terms_beside_spare_vertices_match_oracle(solver, law):
    """Vertices of no element, numbered last: no faces, no slots."""
    print(f"[gpu] viscous spare vertices {law}", flush=True)
    mesh = mg.tri_mesh(6)
    mesh.coord = np.concatenate([mesh.coord, np.random.default_rng(2).random((70, 3))])
    viscous_matches_oracle(solver, mesh, law, {}, {})


def skew_fan_mesh(k, seed, amp):
    """k prisms around an axis in one layer, every vertex displaced: the wall
    faces are not perpendicular to the faces between the prisms."""
    rng = np.random.default_rng(seed)
    ang = 2 * np.pi * np.arange(k) / k + 0.1
    pts = np.concatenate([[[0.0, 0.0]], np.stack([np.cos(ang), np.sin(ang)], 1)])
    bottom = np.column_stack([pts, amp * rng.uniform(-1, 1, k + 1)])
    top = np.column_stack([pts + amp * rng.uniform(-1, 1, pts.shape), 0.8 + amp * rng.uniform(-1, 1, k + 1)])
    q = np.arange(k)
    low = np.stack([0 * q, 1 + q, 1 + (q + 1) % k], 1)
    ev = np.concatenate([low, low + k + 1], 1) + 1
    return mg.Mesh(np.concatenate([bottom, top]), np.full(k, 6, np.int32), ev.astype(np.int32).ravel(),
                   boundary_2d=False, name="skewfan")


def skew_tri_mesh(seed, amp):
    """5^2 squares in prisms, one layer, every vertex displaced."""
    mesh = mg.tri_mesh(5, seed=seed)
    mesh.boundary_2d = False
    mesh.coord = mesh.coord + amp / 5 * np.random.default_rng(seed).uniform(-1, 1, mesh.coord.shape)
    return mesh


# the fraction s of the way from 400 K to cell temperatures of 120 K and 2,500 K
# at which a diagonal pivot of a vertex vanishes in face order (to 1e-15 of its
# row; viscosities up to 4:1 to 8:1), and the largest condition number of a system:
# each size class, 32 lanes, 64 lanes and a workgroup per vertex
@pytest.mark.parametrize("mk,seed,s,cond", [(lambda: skew_tri_mesh(569, 0.25), 569, 0.9366430843065954, 184.5),
                                            (lambda: skew_fan_mesh(5, 521, 0.35), 521, 0.8174891833388135, 92.4),
                                            (lambda: skew_fan_mesh(12, 1397, 0.3), 1397, 0.8620630162572106, 113.2),
                                            (lambda: skew_fan_mesh(24, 307, 0.2), 307, 0.6459062946775922, 270.2)],
                         ids=["tri5", "fan5", "fan12", "fan24"])
def test_vanishing_pivots_under_sutherland_match_oracle(solver, mk, seed, s, cond):
    """Within 1e-12 of the viscous terms' scale or 64 eps times the condition
    number, whichever is larger."""
    mesh = mk()
    print(f"[gpu] viscous skewed {mesh.name} {mesh.n_elems}", flush=True)
    n = mesh.n_elems
    rng = np.random.default_rng(seed + 1000)
    T = 400.0 + s * (np.where(rng.random(n) < 0.5, 120.0, 2500.0) * rng.uniform(0.9, 1.1, n) - 400.0)
    w = np.zeros((n, 5))
    w[:, 0] = 1.0
    w[:, 1:4] = np.random.default_rng(1).uniform(-30, 30, (n, 3))
    w[:, 4] = 0.4 * 720.19471 * T
    viscous_matches_oracle(solver, mesh, "sutherland", dict(boundary_2d=False), {}, mg.primit_to_conserv(w),
                           max(1e-12, 64 * np.finfo(float).eps * cond))


def test_vertices_beyond_the_limit_are_rejected(solver):
    print("[gpu] diffusion limit", flush=True)
    solver.build_mesh(fan_prism_mesh(k=40))  # the axis vertex between the layers has 80 sub-elements
    solver.set_config(make_config("multi_point", boundary_2d=False))
    solver.set_diffusion(True, mu=1e-3)
    solver.put_sol(mg.primit_to_conserv(np.tile([1.0, 0, 0, 0, 1.0], (solver.n_elems, 1))))
    with pytest.raises(SubfvError):
        solver.compute_rhs_ns()
    solver.set_diffusion(False)


def warm_state(xc, seed=3):
    """air-like temperatures (250-350 K) so Sutherland's mu varies by ~30 %"""
    rng = np.random.default_rng(seed)
    x, y = xc[:, 0], xc[:, 1]
    rho = 1.0 + 0.2 * np.sin(3 * x + 1) * np.cos(2 * y) + 0.02 * rng.random(x.size)
    T = 300.0 + 50.0 * np.sin(2 * np.pi * x) * np.cos(np.pi * y) + rng.random(x.size)
    w = np.stack([rho, 30 * np.sin(2 * y + 0.5), -20 * np.cos(3 * x), 5 * np.sin(4 * xc[:, 2] + x),
                  rho * 0.4 * 720.19471 * T], 1)
    return mg.primit_to_conserv(w)


@pytest.mark.parametrize("second", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_sutherland_rhs_and_diag_match_oracle(solver, name, second):
    """compute_mu with use_sutherland: mu per cell, mu0corr their minimum;
    T^1.5 goes through pow on both sides, so the per-cell viscosities may
    differ in the last bit: the same 1e-12 bound as the constant case."""
    print(f"[gpu] sutherland rhs {name} second={second}", flush=True)
    mk, cfgkw, dkw = CASES[name]
    mesh = mk()
    solver.build_mesh(mesh)
    om = O.OracleMesh(mesh)
    sol = warm_state(om.elem_coord)
    solver.set_config(make_config("multi_point", second_order=second, method=4, **cfgkw))
    solver.set_diffusion(True, mu=1.0, **dkw)  # mu_p unused with Sutherland
    solver.set_sutherland(True)
    try:
        solver.put_sol(sol)
        solver.compute_rhs_ns()
        rhs = solver.get("rhs")
        diag = solver.get("diag")
    finally:
        solver.set_sutherland(False)
        solver.set_diffusion(False)
    ocfg = O.make_config("multi_point", second_order=second, method=4, diffusion=True, mu=1.0, sutherland=True,
                         **cfgkw, **dkw)
    mu, mn = O.compute_mu(ocfg, sol)
    assert mu.max() > 1.2 * mn
    r0, sl = om.compute_euler_flux(ocfg, sol)
    if second:
        g = om.compute_cell_grad(sol, 4)[0]
        r2, _ = om.compute_euler_flux(ocfg, sol, grad=g, second_order=True)
        r0 = om.flux_limiting(sol, r0, r2, sl, ocfg.cfl)
    rd, dd = om.add_diffusion(ocfg, sol)
    ref_rhs = r0 + rd
    scale_r = np.abs(rd).max(axis=0) + 1e-300
    assert np.all(np.abs(rhs - ref_rhs) <= 1e-12 * scale_r[None, :] + 1e-14 * np.abs(ref_rhs)), \
        np.abs(rhs - ref_rhs).max(axis=0) / scale_r
    assert np.abs(diag - dd).max() <= 1e-12 * np.abs(dd).max()


def test_sutherland_time_loop_matches_oracle(solver):
    print("[gpu] sutherland run", flush=True)
    mesh = mg.tri_mesh(8)
    solver.build_mesh(mesh)
    om = O.OracleMesh(mesh)
    sol = warm_state(om.elem_coord, 4)
    solver.set_config(make_config("multi_point", second_order=True, method=4, cfl=0.3))
    solver.set_diffusion(True, mu=1.0)
    solver.set_sutherland(True, mu0=1.716e-5, T0=273.15)
    solver.set_time(0.0)
    try:
        solver.put_sol(sol)
        solver.run(10, 0)
        got = solver.get_sol()
    finally:
        solver.set_sutherland(False)
        solver.set_diffusion(False)
    st, ref, info = om.run(O.make_config("multi_point", second_order=True, method=4, cfl=0.3, diffusion=True,
                                         mu=1.0, sutherland=True), sol, 10, 0)
    assert st == 0
    assert np.abs(got - ref).max() / np.abs(ref).max() <= 1e-12
    # the viscous terms moved the state: the same run without them differs
    st, inv, _ = om.run(O.make_config("multi_point", second_order=True, method=4, cfl=0.3), sol, 10, 0)
    assert np.abs(got - inv).max() / np.abs(ref).max() > 1e-9


def test_sutherland_off_restores_constant_viscosity(solver):
    """the blocks formed per residual under Sutherland are replaced by the
    constant-viscosity ones when it is switched off: same bits as before"""
    print("[gpu] sutherland toggle", flush=True)
    mesh = mg.quad_mesh(9)
    solver.build_mesh(mesh)
    sol = warm_state(solver.elem_coord, 6)
    solver.set_config(make_config("multi_point"))
    solver.set_diffusion(True, mu=2e-5)
    solver.put_sol(sol)
    solver.compute_rhs_ns()
    a = solver.get("rhs"), solver.get("diag")
    solver.set_sutherland(True)
    solver.compute_rhs_ns()
    b = solver.get("rhs"), solver.get("diag")
    solver.set_sutherland(False)
    solver.set_diffusion(True, mu=2e-5)
    solver.compute_rhs_ns()
    c = solver.get("rhs"), solver.get("diag")
    solver.set_diffusion(False)
    assert not np.array_equal(a[1], b[1])
    assert np.array_equal(a[0], c[0]) and np.array_equal(a[1], c[1])


def test_viscous_parameter_changes_reuse_the_buffers(solver):
    """Changing mu, toggling Sutherland's law and switching the viscous terms
    off and on re-form the blocks in the buffers of the first viscous
    residual: the context's device memory stays flat."""
    print("[gpu] diffusion parameter sweep memory", flush=True)
    mesh = mg.tri_mesh(12)
    solver.build_mesh(mesh)
    sol = warm_state(solver.elem_coord, 2)
    solver.set_config(make_config("multi_point"))
    solver.put_sol(sol)
    solver.set_diffusion(True, mu=2e-5)
    solver.compute_rhs_ns()
    first = solver.get("rhs")
    solver.set_sutherland(True)  # the per-cell viscosities join the buffers once
    solver.compute_rhs_ns()
    solver.set_sutherland(False)
    used = solver.count("device_bytes_used")
    for k in range(6):
        solver.set_diffusion(True, mu=2e-5 * (1 + k))
        solver.set_sutherland(k % 2 == 1)
        solver.compute_rhs_ns()
        solver.set_diffusion(False)
        solver.compute_rhs_ns()
    solver.set_sutherland(False)
    solver.set_diffusion(True, mu=2e-5)
    solver.compute_rhs_ns()
    assert solver.count("device_bytes_used") == used
    assert np.array_equal(solver.get("rhs"), first)
    solver.set_diffusion(False)


@pytest.mark.parametrize("name", list(CASES))
def test_reference_builders_for_given_viscosities(solver, name):
    """build_momentum_diff_mat_into_global_mat_diag (parts 1) and
    build_diff_mat_into_global_mat_diag (parts 2) for cell viscosities the
    caller gives (varying by a factor 3), each added to a nonzero rhs and
    diag as the reference's builders add them, against the oracle's builders;
    parts 3 is both.  Within 1e-12 of the viscous terms' scale.  A residual
    afterwards uses the constant viscosity again."""
    print(f"[gpu] reference builders {name}", flush=True)
    mk, cfgkw, dkw = CASES[name]
    mesh = mk()
    solver.build_mesh(mesh)
    om = O.OracleMesh(mesh)
    ne = om.n_elems
    sol = smooth_state(om.elem_coord)
    rng = np.random.default_rng(11)
    mu = 2e-3 * (0.5 + rng.random(ne))
    mu0 = float(mu.min())
    rhs0 = rng.standard_normal((ne, 5))
    diag0 = rng.standard_normal((ne, 5, 5))
    solver.set_config(make_config("multi_point", **cfgkw))
    solver.set_diffusion(True, mu=2e-3, **dkw)
    ocfg = O.make_config("multi_point", diffusion=True, mu=2e-3, **cfgkw, **dkw)
    try:
        for parts in (1, 2, 3):
            r, d = solver.add_diffusion(sol, mu, mu0, parts, rhs0, diag0)
            ro, do = om.add_diffusion_mu(ocfg, sol, mu, mu0, parts, rhs0, diag0)
            zr, zd = om.add_diffusion_mu(ocfg, sol, mu, mu0, parts)
            scale_r = np.abs(zr).max() + 1e-300
            scale_d = np.abs(zd).max() + 1e-300
            # the terms land in rhs0 and diag0 in another order: within 1e-12
            # of their scale plus the rounding of those sums
            assert np.all(np.abs(r - ro) <= 1e-12 * scale_r + 1e-14 * np.abs(ro)), (parts, np.abs(r - ro).max())
            assert np.all(np.abs(d - do) <= 1e-12 * scale_d + 1e-14 * np.abs(do)), (parts, np.abs(d - do).max())
            # the rows and blocks a builder does not touch stay as given
            assert np.array_equal(r[:, 0], rhs0[:, 0])
            # (blocks column-major: d[c, j, i] is diag(i + 1, j + 1, c + 1))
            if parts == 1:
                assert np.array_equal(d[:, :, 4], diag0[:, :, 4])  # the heat row diag(5, :)
            if parts == 2:
                assert np.array_equal(r[:, 1:4], rhs0[:, 1:4])
                assert np.array_equal(d[:, 1:4, 1:4], diag0[:, 1:4, 1:4])
        # compute_mu without Sutherland: mu_p everywhere
        m, m0 = solver.compute_mu(sol)
        assert np.all(m == 2e-3) and m0 == 2e-3
        # the context's own residual uses mu_p again
        solver.put_sol(sol)
        solver.compute_rhs_ns()
        rd, dd = om.add_diffusion(ocfg, sol)
        r0, _ = om.compute_euler_flux(ocfg, sol)
        scale_r = np.abs(rd).max(axis=0) + 1e-300
        assert np.all(np.abs(solver.get("rhs") - (r0 + rd)) <= 1e-12 * scale_r[None, :] + 1e-14 * np.abs(r0 + rd))
    finally:
        solver.set_diffusion(False)


def test_compute_mu_sutherland_matches_oracle(solver):
    """compute_mu with use_sutherland: per-cell viscosities and mu0corr (their
    minimum); T^1.5 goes through pow on both sides: within 4 ulp."""
    print("[gpu] compute_mu sutherland", flush=True)
    mesh = mg.tri_mesh(9)
    solver.build_mesh(mesh)
    om = O.OracleMesh(mesh)
    sol = warm_state(om.elem_coord, 3)
    solver.set_config(make_config("multi_point"))
    solver.set_diffusion(True, mu=1.0)
    solver.set_sutherland(True)
    try:
        m, m0 = solver.compute_mu(sol)
        # the builders on these viscosities: the context's Sutherland residual
        r, d = solver.add_diffusion(sol, m, m0, 3)
    finally:
        solver.set_sutherland(False)
        solver.set_diffusion(False)
    ocfg = O.make_config("multi_point", diffusion=True, mu=1.0, sutherland=True)
    mo, m0o = O.compute_mu(ocfg, sol)
    assert mo.max() > 1.2 * m0o
    assert np.abs(m - mo).max() <= 4 * np.spacing(mo).max()
    assert abs(m0 - m0o) <= 4 * np.spacing(m0o)
    rd, dd = om.add_diffusion(ocfg, sol)
    assert np.abs(r - rd).max() <= 1e-12 * np.abs(rd).max()
    assert np.abs(d - dd).max() <= 1e-12 * np.abs(dd).max()


_MEMINFO = """
#include <stddef.h>
size_t free_now = 0;  /* 0: plenty */
int hipMemGetInfo(size_t *f, size_t *t) {
  *t = (size_t)1 << 38;
  *f = free_now ? free_now : *t;
  return 0;
}
"""

_RETRY = """
import ctypes, sys
sys.path[:0] = {path!r}
info = ctypes.CDLL({so!r}, mode=ctypes.RTLD_GLOBAL)  # before the library, whose calls it answers
free_now = ctypes.c_size_t.in_dll(info, "free_now")
import numpy as np
from subfv_amd import meshgen as mg
from subfv_amd.api import Solver, SubfvError, make_config
from test_gpu_diffusion import smooth_state

def rhs(s, sol):
    s.put_sol(sol)
    s.compute_rhs_ns()
    return s.get("rhs")

s = Solver(0)
s.build_mesh(mg.tri_mesh(60))
s.set_config(make_config("multi_point"))
s.set_diffusion(True, mu=2e-3)
sol = smooth_state(s.elem_coord)
used = s.count("device_bytes_used")
V, SF, SE, C = s.n_vert, s.n_sub_faces, s.n_sub_elems, s.n_elems
# room for the tables and the work arrays, not for the inverses behind them
free_now.value = (1 << 30) + 4 * V + SF + 12 * SE + 8 * (V + 16 * SE + 39 * C) + (1 << 20)
for _ in range(3):
    try:
        rhs(s, sol)
        raise AssertionError("accepted")
    except SubfvError as e:
        assert "MiB needed" in str(e), e
    # (the work arrays of the inviscid residual before it aside)
    held = s.count("device_bytes_used")
    first = locals().get("first", held)
    assert held == first, (held, first)
free_now.value = 0
got = rhs(s, sol)
grown = s.count("device_bytes_used")
t = Solver(0)
t.build_mesh(mg.tri_mesh(60))
t.set_config(make_config("multi_point"))
t.set_diffusion(True, mu=2e-3)
assert np.array_equal(rhs(t, sol), got)
assert t.count("device_bytes_used") == grown, (t.count("device_bytes_used"), grown)
print("RETRY_OK", used, first, grown)
"""


def test_failed_viscous_setup_takes_nothing(tmp_path):
    """Viscous residuals refused for want of device memory, after the tables
    were formed: each attempt gives back what it took, and with room again the
    residual and the memory held are those of a context that never failed."""
    print("[gpu] viscous setup without room", flush=True)
    src, so = tmp_path / "meminfo.c", tmp_path / "libmeminfo.so"
    src.write_text(_MEMINFO)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    here = os.path.dirname(os.path.abspath(__file__))
    path = [os.path.dirname(here), here, os.path.join(os.path.dirname(here), "oracle")]
    out = subprocess.run([sys.executable, "-c", _RETRY.format(path=path, so=str(so))], capture_output=True, text=True,
                         timeout=100)
    assert out.returncode == 0 and "RETRY_OK" in out.stdout, out.stdout + out.stderr
