"""Workloads that the explicit force step is timed on, through its Python entry points.

A case names a mesh, a material, a formulation and how many steps one call advances; the
sizes are those of this repository's benchmark and tests (the 6M-Tet4 block, the Taylor bars,
the 20^3 Hex8 cube, the 64^3 RKPM lattice, the uneven Hex8 ensemble, the adjoint block, thex
nodal cells) and generic ones between them.

  listed()             the standing cases
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  solver with mesh, material and initial state, output arrays on the GPU
  run(state)           one pass: steps (or one force evaluation, gradient, ...) and the fields
  work(case)           bytes and flops one pass cannot do without
  exact(case, seed)    the same pass as plain float64 torch gives it
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "aperi-mech_amd", "python"))

import aperi_hip as A  # noqa: E402

STEEL = dict(rho=7850.0, E=200e9, nu=0.3)
SOFT_ALUMINIUM = dict(rho=2700.0, E=70e9, nu=0.33, sy=30e6, hard=1e9)  # yields within the first steps
POLYMER = dict(rho=2700.0, E=78.2e8, nu=0.3)  # the thex bars
MATERIALS = {"le": (A.LINEAR_ELASTIC, STEEL), "nh": (A.NEO_HOOKEAN, STEEL), "svk": (A.SVK, STEEL),
             "j2": (A.J2, SOFT_ALUMINIUM)}


def listed():
    return [
        # a large solid run between two outputs: the 6M-Tet4 block
        dict(name="tet4 block 6M", kind="fem", elem="tet4", nx=100, ny=100, nz=100, mat="nh", form="total",
             fixed=False, calls=1, steps=20),
        # Taylor bars: the smallest mesh, many steps in one call ...
        dict(name="taylor bar 6k", kind="fem", elem="tet4", nx=7, ny=7, nz=21, mat="svk", form="total", fixed=True,
             calls=1, steps=50),
        # ... and the middle one under a time stepper that asks for an increment before every step
        dict(name="taylor bar 49k stepper", kind="fem", elem="tet4", nx=14, ny=14, nz=42, mat="svk", form="total",
             fixed=True, calls=20, steps=1),
        # the plain Hex8 cube, bottom face held
        dict(name="hex8 cube 8k", kind="fem", elem="hex8", nx=20, ny=20, nz=20, mat="nh", form="total", fixed=True,
             calls=1, steps=50),
        # large deformation with plasticity: updated Lagrangian Hex8
        dict(name="hex8 updated j2 33k", kind="fem", elem="hex8", nx=32, ny=32, nz=32, mat="j2", form="updated",
             fixed=False, calls=1, steps=20),
        # the force alone, called by a solver that keeps its own fields on the device
        dict(name="tet4 force 384k", kind="force", elem="tet4", nx=40, ny=40, nz=40, mat="j2"),
        # meshfree: the 64^3-node lattice, the default one-pass force, and a smaller two-pass one
        dict(name="rkpm one-pass 64", kind="rkpm", nx=63, ny=63, nz=63, one_pass=True, scale=1.5, steps=10),
        dict(name="rkpm two-pass 40", kind="rkpm", nx=39, ny=39, nz=39, one_pass=False, scale=1.5, steps=25),
        # nodal cells with F-bar on a thex mesh
        dict(name="nodal f-bar 41k", kind="nodal", nx=12, ny=12, nz=12, scale=0.8, f_bar=True, steps=20),
        # a parameter study: uneven Hex8 specimens stepped together, replayed from a graph
        dict(name="hex8 ensemble 64", kind="ensemble", specimens=64, lo=8, hi=48, mat="nh", steps=10),
        # calibration: gradient of a displacement misfit in E, nu and the initial velocity
        dict(name="adjoint 14k", kind="adjoint", elem="hex8", nx=24, ny=24, nz=24, mat="nh", steps=40, interval=10),
        # the power-method time stepper: a new increment, then the steps until the next one
        dict(name="power stepper 197k", kind="power", elem="tet4", nx=32, ny=32, nz=32, mat="nh", steps=10),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dims(rng, lo, hi, most):
    while True:
        d = [_log(rng, lo, hi) for _ in range(3)]
        if d[0] * d[1] * d[2] <= most:
            return dict(nx=d[0], ny=d[1], nz=d[2])


def draw(rng):
    kind = rng.choice(["fem", "fem", "fem", "fem", "force", "rkpm", "rkpm", "nodal", "ensemble", "adjoint", "power"])
    if kind == "fem":
        elem = rng.choice(["tet4", "tet4", "hex8"])
        form = rng.choice(["total", "total", "total", "updated", "semi"])
        most = 200_000 if elem == "tet4" else 120_000
        d = _dims(rng, 5, 90, most if form == "total" else most // 4)
        calls, steps = (1, _log(rng, 2, 40)) if rng.random() < 0.7 else (rng.randint(2, 16), 1)
        return dict(kind=kind, elem=elem, **d, mat=rng.choice(["le", "nh", "svk", "j2"]), form=form,
                    fixed=rng.random() < 0.5, calls=calls, steps=steps)
    if kind == "force":
        elem = rng.choice(["tet4", "hex8"])
        return dict(kind=kind, elem=elem, **_dims(rng, 5, 70, 150_000), mat=rng.choice(["le", "nh", "svk", "j2"]))
    if kind == "rkpm":
        return dict(kind=kind, **_dims(rng, 6, 50, 60_000), one_pass=rng.random() < 0.6,
                    scale=round(rng.uniform(1.05, 1.6), 2), steps=_log(rng, 2, 20))
    if kind == "nodal":
        f_bar = rng.random() < 0.6
        return dict(kind=kind, **_dims(rng, 4, 16, 2000), scale=0.8 if f_bar else 0.9, f_bar=f_bar,
                    steps=_log(rng, 2, 30))
    if kind == "ensemble":
        return dict(kind=kind, specimens=_log(rng, 4, 64), lo=6, hi=rng.randint(12, 36), mat=rng.choice(["le", "nh"]),
                    steps=2 * _log(rng, 2, 10))
    if kind == "adjoint":
        return dict(kind=kind, elem=rng.choice(["hex8", "tet4"]), **_dims(rng, 5, 24, 8000),
                    mat=rng.choice(["le", "nh"]), steps=rng.randint(8, 40), interval=rng.randint(4, 12))
    return dict(kind="power", elem=rng.choice(["tet4", "hex8"]), **_dims(rng, 6, 48, 40_000),
                mat=rng.choice(["le", "nh", "svk"]), steps=_log(rng, 2, 20))


# ---------------- meshes and initial states (host, from the seed alone) ----------------

_KUHN = [(0, 1, 2, 6), (0, 5, 1, 6), (0, 2, 3, 6), (0, 3, 7, 6), (0, 4, 5, 6), (0, 7, 4, 6)]


@functools.lru_cache(maxsize=4)
def _lattice(nx, ny, nz):
    """Unjittered node positions (cell edge 1 / max(n)) and Hex8 connectivity, x fastest."""
    n = max(nx, ny, nz)
    k, j, i = np.meshgrid(np.arange(nz + 1), np.arange(ny + 1), np.arange(nx + 1), indexing="ij")
    X = np.stack([i.ravel(), j.ravel(), k.ravel()], axis=1) / float(n)
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    i, j, k = i.ravel(), j.ravel(), k.ravel()
    node = lambda a, b, c: (i + a) + (nx + 1) * ((j + b) + (ny + 1) * (k + c))  # noqa: E731
    conn = np.stack([node(0, 0, 0), node(1, 0, 0), node(1, 1, 0), node(0, 1, 0),
                     node(0, 0, 1), node(1, 0, 1), node(1, 1, 1), node(0, 1, 1)], axis=1).astype(np.int32)
    return X, conn


@functools.lru_cache(maxsize=2)
def _tets(nx, ny, nz):
    _, hexes = _lattice(nx, ny, nz)
    return np.stack([hexes[:, list(t)] for t in _KUHN], axis=1).reshape(-1, 4)


@functools.lru_cache(maxsize=4)
def _thex(nx, ny, nz):
    """Four hexes per tet: the vertex, its three edge midpoints, face centroids, the tet's centroid."""
    tets = _tets(nx, ny, nz).astype(np.int64)
    nv = (nx + 1) * (ny + 1) * (nz + 1)
    epairs, fpairs = [(0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3)], [(0, 1, 2), (0, 1, 3), (0, 2, 3), (1, 2, 3)]
    edges, ei = np.unique(np.sort(tets[:, epairs].reshape(-1, 2), axis=1), axis=0, return_inverse=True)
    faces, fi = np.unique(np.sort(tets[:, fpairs].reshape(-1, 3), axis=1), axis=0, return_inverse=True)
    ei, fi = ei.reshape(-1, 6) + nv, fi.reshape(-1, 4) + nv + len(edges)
    cen = nv + len(edges) + len(faces) + np.arange(len(tets))
    e = {p: ei[:, k] for k, p in enumerate(epairs)}
    f = {p: fi[:, k] for k, p in enumerate(fpairs)}
    out = []
    for v in range(4):
        a, b, c = [k for k in range(4) if k != v]
        if v in (1, 3):  # (a, b, c) seen from v is right-handed for v = 0 and 2 of a positive tet
            b, c = c, b
        E = lambda p, q: e[tuple(sorted((p, q)))]  # noqa: E731
        F = lambda p, q, r: f[tuple(sorted((p, q, r)))]  # noqa: E731
        out.append(np.stack([tets[:, v], E(v, a), F(v, a, b), E(v, b), E(v, c), F(v, a, c), cen, F(v, b, c)], axis=1))
    return tets, edges, faces, np.stack(out, axis=1).reshape(-1, 8).astype(np.int32)


def _mesh(case, seed, elem):
    """Jittered lattice (10 % of the cell edge) as hexes or Kuhn tets; its cell edge."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    X, hexes = _lattice(nx, ny, nz)
    h = 1.0 / max(nx, ny, nz)
    X = X + 0.1 * h * np.random.default_rng([seed, 1]).uniform(-1.0, 1.0, X.shape)
    return X, (hexes if elem == "hex8" else _tets(nx, ny, nz)), h


def _lame(E, nu):
    return E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))


def _dt(h, mat, elem):
    """Half the wave transit bound of the jittered cell or Kuhn tet (thex: of its short edges)."""
    lam, mu = _lame(mat["E"], mat["nu"])
    return {"hex8": 0.35, "tet4": 0.15, "thex": 0.05}[elem] * h / math.sqrt((lam + 2 * mu) / mat["rho"])


def _velocity(X, seed, ramp=0.0):
    """0.5 m/s of noise per component; plastic runs add a stretching ramp about the centre."""
    v = 0.5 * np.random.default_rng([seed, 2]).standard_normal(X.shape)
    return v + ramp * (X - X.mean(axis=0)) * np.array([-0.5, -0.5, 1.0])


def _problem(case, seed):
    """Host arrays and numbers of a single-block case."""
    elem = case.get("elem", "tet4")
    if case["kind"] == "nodal":
        X, _, h = _mesh(case, seed, "tet4")
        tets, edges, faces, conn = _thex(case["nx"], case["ny"], case["nz"])
        X = np.concatenate([X, X[edges].mean(axis=1), X[faces].mean(axis=1), X[tets].mean(axis=1)])
        kind, mat, ramp, elem = A.SVK, POLYMER, 5.0, "thex"
    else:
        X, conn, h = _mesh(case, seed, elem)
        kind, mat = MATERIALS[case.get("mat", "j2")]
        ramp = 100.0 if kind == A.J2 else 0.0
    v = _velocity(X, seed, ramp)
    fixed = None
    if case.get("fixed"):
        fixed = np.zeros(X.shape, dtype=np.uint8)
        fixed[X[:, 2] < 0.5 * h] = 1
        v[fixed.astype(bool)] = 0.0
    return dict(X=X, conn=conn, h=h, kind=kind, mat=mat, v=v, fixed=fixed, dt=_dt(h, mat, elem),
                etype=A.TET4 if elem == "tet4" else A.HEX8)


def _specimens(case, seed):
    """Uneven Hex8 cubes, edges log-uniform in [lo, hi], own E, nu and time increment."""
    r = np.random.default_rng([seed, 3])
    # one edge count per quantile, so that every seed's ensemble has the same size
    q = (np.arange(case["specimens"]) + 0.5) / case["specimens"]
    edges = np.rint(np.exp(math.log(case["lo"]) + q * math.log(case["hi"] / case["lo"]))).astype(int)
    out = []
    for n in r.permutation(edges):
        X, conn = _lattice(int(n), int(n), int(n))
        mat = dict(rho=7850.0, E=r.uniform(50e9, 250e9), nu=r.uniform(0.2, 0.45))
        out.append(dict(X=X, conn=conn, mat=mat, dt=_dt(1.0 / n, mat, "hex8"), v=r.uniform(-1.0, 1.0, X.shape)))
    return out


def _parameter_fields(case, p, seed):
    """Per-element E and nu (smooth waves about the block's values) and the target displacement."""
    r = np.random.default_rng([seed, 4])
    cen = p["X"][p["conn"]].mean(axis=1)
    wave = lambda: np.cos(cen @ r.normal(0.0, 5.0, 3) + r.uniform(0.0, 2 * math.pi))  # noqa: E731
    return 200e9 * (1 + 0.15 * wave()), 0.3 + 0.04 * wave(), 1e-6 * r.standard_normal(p["X"].shape)


# ---------------- prepare and run ----------------

_SHAPE = {"u": 3, "v": 3, "a": 3, "f": 3, "H": 9, "P": 9, "state": 0}
_FIELD = {"u": A.FIELD_U, "v": A.FIELD_V, "a": A.FIELD_A, "f": A.FIELD_F, "H": A.FIELD_H, "P": A.FIELD_P,
          "state": A.FIELD_STATE}


def _outputs(names, nn, ne):
    """Device arrays that the fields are read into."""
    n = {k: nn if k in "uvaf" else ne for k in names}
    shape = {k: (n[k], _SHAPE[k]) if _SHAPE[k] else (n[k],) for k in names}
    return {k: torch.zeros(shape[k], dtype=torch.float64, device="cuda") for k in names}


def _read(s, out):
    for k, t in out.items():
        s.get_field_device(_FIELD[k], t.data_ptr())
    return out


def prepare(case, seed):
    torch.cuda.init()
    kind = case["kind"]
    s = A.Solver()
    if kind == "ensemble":
        specs = _specimens(case, seed)
        s.batch_begin(A.HEX8, MATERIALS[case["mat"]][0])
        for sp in specs:
            s.batch_add(sp["X"], sp["conn"], sp["mat"]["rho"], sp["mat"]["E"], sp["mat"]["nu"], sp["dt"])
        s.batch_end()
        s.compute_mass()
        s.set_field(A.FIELD_V, np.concatenate([sp["v"] for sp in specs]))
        s.initialize()
        s.set_graph(True)
        return dict(case=case, s=s, out=_outputs("u v a f H P".split(), s.nn, s.ne))
    p = _problem(case, seed)
    m = p["mat"]
    s.set_mesh(p["etype"], p["X"], p["conn"])
    s.set_material(p["kind"], m["rho"], m["E"], m["nu"], m.get("sy", 0.0), m.get("hard", 0.0))
    if kind == "rkpm":
        s.rk_setup(case["scale"], one_pass=case["one_pass"])
    elif kind == "nodal":
        s.rk_nodal_setup(case["scale"], 0 if case["f_bar"] else 1, case["f_bar"])
    elif case.get("form") == "updated":
        s.set_formulation(A.UPDATED_LAGRANGIAN)
    elif case.get("form") == "semi":
        s.set_semi_lagrangian(5)
    s.compute_mass()
    if p["fixed"] is not None:
        s.set_fixed(p["fixed"])
    names = "u v a f H P".split() + (["state"] if p["kind"] == A.J2 else [])
    state = dict(case=case, s=s, dt=p["dt"])
    if kind == "adjoint":
        E, nu, target = _parameter_fields(case, p, seed)
        return dict(state, E=E, nu=nu, target=target, v0=p["v"], u0=np.zeros_like(p["X"]))
    if kind == "force":  # displacements of the size the ramp reaches in some dozens of steps
        u = _velocity(p["X"], seed, 100.0) * 30 * p["dt"]
        names = "f H P".split() + (["state"] if p["kind"] == A.J2 else [])
        state["u"] = torch.from_numpy(u).cuda()
    else:
        s.set_field(A.FIELD_V, p["v"])
        s.initialize()
    if kind == "nodal":
        names = "u v a f".split()  # element fields of nodal cells have no device transfer
    state["out"] = _outputs(names, s.nn, s.ne)
    if kind == "power":
        state["last"] = 0.0
    return state


def run(state):
    case, s = state["case"], state["s"]
    kind = case["kind"]
    if kind == "adjoint":
        s.set_material_fields(state["E"], state["nu"])
        s.set_field(A.FIELD_U, state["u0"])
        s.set_field(A.FIELD_V, state["v0"])
        s.initialize()
        s.adjoint_forward(state["dt"], case["steps"], case["interval"])
        u = s.get(A.FIELD_U)
        E_bar, nu_bar, v0_bar = s.adjoint_backward(u - state["target"])
        return dict(u=u, E_bar=E_bar, nu_bar=nu_bar, v0_bar=v0_bar)
    if kind == "force":
        s.set_field_device(A.FIELD_U, state["u"].data_ptr())
        s.internal_force(0.0, state["dt"])
        return _read(s, state["out"])
    if kind == "power":
        full, iterations, converged = s.power_method_time_increment(previous_time_increment=state["last"])
        state["last"] = full
        s.step(0.5 * full, case["steps"])
        return dict(_read(s, state["out"]), increment=full, iterations=iterations, converged=converged)
    if kind == "ensemble":
        s.step(0.0, case["steps"])
        return _read(s, state["out"])
    for _ in range(case.get("calls", 1)):
        s.step(state["dt"], case["steps"])
    return _read(s, state["out"])


# ---------------- work ----------------

def work(case):
    """Mesh, node state and parameters read once, fields written once; multiply-adds of the
    element evaluations (about 550 flops a Tet4, 5300 a Hex8, 2300 a smoothed thex hex)."""
    kind = case["kind"]
    if kind == "ensemble":
        e = [len(sp["conn"]) for sp in _specimens(case, 0)]
        n = [len(sp["X"]) for sp in _specimens(case, 0)]
        ne, nn = float(sum(e)), float(sum(n))
        return {"bytes": ne * (32 + 16 + 144) + nn * 208, "flops": 5300 * ne * case["steps"]}
    cells = float(case["nx"] * case["ny"] * case["nz"])
    nn = float((case["nx"] + 1) * (case["ny"] + 1) * (case["nz"] + 1))
    if kind == "nodal":
        ne = 24 * cells
        # the neighbor values of every thex node (about 12 cells of nodes, 20 neighbors each)
        return {"bytes": ne * (32 + 144) + nn * 200 + 25 * nn * 20 * 12, "flops": 2300 * ne * case["steps"]}
    npe = 8 if case.get("elem") == "hex8" else 4
    ne = cells if npe == 8 else 6 * cells
    flops = 5300 if npe == 8 else 550
    state = 16 if case.get("mat", "j2") == "j2" else 0
    if kind == "rkpm":  # the functions (id and value of up to 40 neighbors a node) instead of their products
        return {"bytes": ne * (16 + 144 + 16) + nn * (200 + 40 * 12), "flops": (550 * ne + 320 * nn) * case["steps"]}
    if kind == "force":
        return {"bytes": ne * (4 * npe + 144 + state) + nn * 72, "flops": flops * ne}
    if kind == "adjoint":  # forward, recomputed forward and the reverse step (about three forwards)
        return {"bytes": ne * (4 * npe + 32) + nn * 160, "flops": 5 * flops * ne * case["steps"]}
    if kind == "power":  # about ten force evaluations for the increment
        return {"bytes": ne * (4 * npe + 144) + nn * 232, "flops": flops * ne * (case["steps"] + 10)}
    return {"bytes": ne * (4 * npe + 144 + state) + nn * 200,
            "flops": flops * ne * case["steps"] * case["calls"]}


# ---------------- the same passes in plain float64 torch ----------------
# 3x3 tensors are nested lists of one value per element.

def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a)).to(_dev())


def _mm(P, Q):
    return [[P[i][0] * Q[0][j] + P[i][1] * Q[1][j] + P[i][2] * Q[2][j] for j in range(3)] for i in range(3)]


def _tr(P):
    return [[P[j][i] for j in range(3)] for i in range(3)]


def _inv(M):
    c = [[M[(j + 1) % 3][(i + 1) % 3] * M[(j + 2) % 3][(i + 2) % 3] - M[(j + 1) % 3][(i + 2) % 3] * M[(j + 2) % 3][(i + 1) % 3]
          for j in range(3)] for i in range(3)]
    det = M[0][0] * c[0][0] + M[0][1] * c[1][0] + M[0][2] * c[2][0]
    return [[c[i][j] / det for j in range(3)] for i in range(3)], det


def _plus_i(M):
    return [[M[i][j] + 1.0 if i == j else M[i][j] for j in range(3)] for i in range(3)]


def _jm1(H):
    """det(I + H) - 1 by the invariants of H."""
    i2 = (H[0][0] * H[1][1] - H[0][1] * H[1][0] + H[0][0] * H[2][2] - H[0][2] * H[2][0]
          + H[1][1] * H[2][2] - H[1][2] * H[2][1])
    return H[0][0] + H[1][1] + H[2][2] + i2 + (
        H[0][0] * (H[1][1] * H[2][2] - H[1][2] * H[2][1]) - H[0][1] * (H[1][0] * H[2][2] - H[1][2] * H[2][0])
        + H[0][2] * (H[1][0] * H[2][1] - H[1][1] * H[2][0]))


def _stress(kind, H, lam, mu, mat, ep):
    """First Piola-Kirchhoff stress and the new equivalent plastic strain."""
    I3 = range(3)
    if kind in (A.LINEAR_ELASTIC, A.J2):
        eps = [[0.5 * (H[i][j] + H[j][i]) for j in I3] for i in I3]
        t = eps[0][0] + eps[1][1] + eps[2][2]
        if kind == A.LINEAR_ELASTIC:
            return [[2 * mu * eps[i][j] + (lam * t if i == j else 0.0) for j in I3] for i in I3], ep
        dev = [[2 * mu * (eps[i][j] - (t / 3 if i == j else 0.0)) for j in I3] for i in I3]
        norm = torch.sqrt(sum(dev[i][j] ** 2 for i in I3 for j in I3))
        phi = math.sqrt(1.5) * norm - (mat["sy"] + mat["hard"] * ep)
        dep = torch.where(phi > 0, phi / (3 * mu + mat["hard"]), torch.zeros_like(phi))
        keep = 1 - torch.where(phi > 0, math.sqrt(6.0) * mu * dep / norm, torch.zeros_like(phi))
        K = lam + 2 * mu / 3
        return [[dev[i][j] * keep + (K * t if i == j else 0.0) for j in I3] for i in I3], ep + dep
    F = _plus_i(H)
    if kind == A.SVK:
        hth = _mm(_tr(H), H)
        G = [[0.5 * (H[i][j] + H[j][i] + hth[i][j]) for j in I3] for i in I3]
        t = G[0][0] + G[1][1] + G[2][2]
        return _mm(F, [[2 * mu * G[i][j] + (lam * t if i == j else 0.0) for j in I3] for i in I3]), ep
    hht = _mm(H, _tr(H))
    lnJ = torch.log1p(_jm1(H))
    tau = [[mu * (hht[i][j] + H[i][j] + H[j][i]) + (lam * lnJ if i == j else 0.0) for j in I3] for i in I3]
    return _mm(tau, _tr(_inv(F)[0])), ep


_CORNER = np.array([[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1], [-1, -1, 1], [1, -1, 1], [1, 1, 1], [-1, 1, 1]])
_FACES = [(0, 1, 5, 4), (1, 2, 6, 5), (2, 3, 7, 6), (0, 4, 7, 3), (0, 3, 2, 1), (4, 5, 6, 7)]


def _corners(x, conn):
    return [x[conn[:, k]].unbind(1) for k in range(conn.shape[1])]


def _points(etype, X):
    """(B[k][j], weight) of every integration point for corner positions X[k][d]."""
    if etype == A.TET4:
        Ji, det = _inv([[X[j + 1][i] - X[0][i] for j in range(3)] for i in range(3)])
        B = [[-Ji[0][j] - Ji[1][j] - Ji[2][j] for j in range(3)]] + [list(Ji[k]) for k in range(3)]
        yield B, det / 6
        return
    for q in _CORNER / math.sqrt(3.0):
        f = 1 + _CORNER * q
        dN = np.stack([_CORNER[:, 0] * f[:, 1] * f[:, 2], _CORNER[:, 1] * f[:, 0] * f[:, 2],
                       _CORNER[:, 2] * f[:, 0] * f[:, 1]], axis=1) / 8
        Ji, det = _inv([[sum(X[k][i] * float(dN[k, d]) for k in range(8)) for d in range(3)] for i in range(3)])
        yield [[sum(float(dN[k, d]) * Ji[d][j] for d in range(3)) for j in range(3)] for k in range(8)], det


def _smoothed_hex(X):
    """Face-smoothed gradient and volume of a hex, every face split about its centroid."""
    B, V = [[0.0, 0.0, 0.0] for _ in range(8)], 0.0
    for face in _FACES:
        mid = [sum(X[k][d] for k in face) / 4 for d in range(3)]
        for k in range(4):
            p, q = [X[face[k - 1]][d] - mid[d] for d in range(3)], [X[face[k]][d] - mid[d] for d in range(3)]
            n = [(p[(d + 1) % 3] * q[(d + 2) % 3] - p[(d + 2) % 3] * q[(d + 1) % 3]) / 2 for d in range(3)]
            V = V + sum(mid[d] * n[d] for d in range(3)) / 3
            for m in range(4):
                c = (5 if m in (k, (k - 1) % 4) else 1) / 12
                B[face[m]] = [B[face[m]][d] + c * n[d] for d in range(3)]
    return [[b / V for b in row] for row in B], V


def _grad(u, B):
    return [[sum(u[k][i] * B[k][j] for k in range(len(B))) for j in range(3)] for i in range(3)]


def _scatter(f, conn, B, P, w):
    """f_k -= w P B_k"""
    for k in range(conn.shape[1]):
        f.index_add_(0, conn[:, k], torch.stack(
            [-w * (P[i][0] * B[k][0] + P[i][1] * B[k][1] + P[i][2] * B[k][2]) for i in range(3)], dim=1))


def _rows(M):
    return torch.stack([M[i][j] for i in range(3) for j in range(3)], dim=1)


def _force(p, u, ep, x=None, Hr=None):
    """f, H, P and the plastic strain; with Hr over the configuration x (u: the increment since)."""
    conn = p["tconn"]
    Xe, Ue = _corners(p["tX"] if x is None else x, conn), _corners(u, conn)
    f = torch.zeros_like(p["tX"])
    for B, w in _points(p["etype"], Xe):
        H = _grad(Ue, B)
        if Hr is not None:
            dd = _mm(H, Hr)
            H = [[H[i][j] + Hr[i][j] + dd[i][j] for j in range(3)] for i in range(3)]
        P, new = _stress(p["kind"], H, p["lam"], p["mu"], p["mat"], ep)
        Q = P
        if Hr is not None:
            Fr = _plus_i(Hr)
            Q, det = _mm(P, _tr(Fr)), _inv(Fr)[1]
            Q = [[Q[i][j] / det for j in range(3)] for i in range(3)]
        _scatter(f, conn, B, Q, w)
    return f, H, P, new


def _lumped(p):
    m = torch.zeros(len(p["tX"]), dtype=torch.float64, device=_dev())
    V = sum(w for _, w in _points(p["etype"], _corners(p["tX"], p["tconn"])))
    for k in range(p["tconn"].shape[1]):
        m.index_add_(0, p["tconn"][:, k], V * p["mat"]["rho"] / p["tconn"].shape[1])
    return m


def _on_device(p):
    lam, mu = _lame(p["mat"]["E"], p["mat"]["nu"])
    free = torch.ones(p["X"].shape, dtype=torch.float64, device=_dev())
    if p["fixed"] is not None:
        free[_t(p["fixed"]).bool()] = 0.0
    return dict(p, tX=_t(p["X"]), tconn=_t(p["conn"]).long(), lam=lam, mu=mu, free=free)


def _march(p, m, steps, force, v, dt, u=None, a=None, after=None):
    """Central differences from (u, v, a); force(u, increment) -> f and what else it gives."""
    u = torch.zeros_like(v) if u is None else u
    if a is None:
        a = force(u, torch.zeros_like(u), 0.0)[0] / m[:, None]
    got = None
    for n in range(steps):
        v = (v + 0.5 * dt * a) * p["free"]
        u = u + dt * v
        got = force(u, dt * v, dt)
        a = got[0] / m[:, None] * p["free"]
        v = v + 0.5 * dt * a
        if after:
            after(n + 1, got)
    return dict(u=u, v=v, a=a, f=got[0]), got


def _fem(case, p):
    m, ep = _lumped(p), torch.zeros(len(p["tconn"]), dtype=torch.float64, device=_dev())
    zero = [[torch.zeros_like(ep)] * 3 for _ in range(3)]
    st = dict(ep=ep, x=p["tX"].clone(), Hr=zero, acc=torch.zeros_like(p["tX"]))
    form = case.get("form", "total")

    def force(u, inc, dt):
        if form == "total":
            got = _force(p, u, st["ep"])
        elif form == "updated":
            got = _force(p, inc, st["ep"], st["x"], st["Hr"])
            st["x"], st["Hr"] = st["x"] + inc, got[1]
        else:
            st["acc"] = st["acc"] + inc
            got = _force(p, st["acc"], st["ep"], st["x"], st["Hr"])
        if dt:
            st["ep"] = got[3]
        return got

    def after(n, got):
        if form == "semi" and n % 5 == 0:
            st["x"], st["acc"], st["Hr"] = st["x"] + st["acc"], torch.zeros_like(st["acc"]), got[1]

    out, got = _march(p, m, case["steps"] * case.get("calls", 1), force, _t(p["v"]), p["dt"], after=after)
    out.update(H=_rows(got[1]), P=_rows(got[2]))
    if p["kind"] == A.J2:
        out["state"] = st["ep"]
    return out


def _max_edge(p, active):
    """Longest edge of the elements around every node; edges to inactive nodes count twice."""
    X, conn = p["tX"], p["tconn"]
    l = torch.zeros(len(X), dtype=torch.float64, device=_dev())
    for a in range(conn.shape[1]):
        for b in range(conn.shape[1]):
            d = (X[conn[:, a]] - X[conn[:, b]]).norm(dim=1) * torch.where(conn[:, b] < active, 1.0, 2.0)
            l.scatter_reduce_(0, conn[:, a], d, "amax")
    return l


def _functions(p, case, active):
    """Neighbors (40 nearest whose ball holds the node) and reproducing-kernel values, rows of 40."""
    X = p["tX"]
    s = case["scale"]
    R = _max_edge(p, active) * (s if s != 1.0 else 1.0 + 1e-6)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    lattice = case["kind"] == "rkpm"
    reach = int(math.ceil(float(R.max()) * 1.05 / p["h"] + 0.2)) if lattice else 0
    ids, vals = [], []
    chunk = max(256, int(2e7 / ((2 * reach + 1) ** 3 if lattice else active)))
    off = torch.arange(-reach, reach + 1, device=_dev())
    for b in range(0, len(X), chunk):
        i = torch.arange(b, min(b + chunk, len(X)), device=_dev())
        if lattice:
            ax = [i % (nx + 1), (i // (nx + 1)) % (ny + 1), i // ((nx + 1) * (ny + 1))]
            g = [ax[d][:, None] + off[None, :] for d in range(3)]
            ok = [(g[d] >= 0) & (g[d] <= n) for d, n in enumerate((nx, ny, nz))]
            j = (g[0][:, None, None, :] + (nx + 1) * (g[1][:, None, :, None] + (ny + 1) * g[2][:, :, None, None]))
            good = (ok[0][:, None, None, :] & ok[1][:, None, :, None] & ok[2][:, :, None, None]).reshape(len(i), -1)
            j = torch.where(good, j.reshape(len(i), -1), torch.zeros((), dtype=torch.int64, device=_dev()))
        else:
            j = torch.arange(active, device=_dev())[None, :].expand(len(i), -1)
            good = torch.ones(j.shape, dtype=torch.bool, device=_dev())
        tweak = torch.tensor([1 + 1e-6, 1 + 1e-7, 1 + 1e-8], dtype=torch.float64, device=_dev())
        d2 = ((X[j] - X[i][:, None, :]) ** 2).sum(dim=2)
        near = ((X[j] * tweak - X[i][:, None, :]) ** 2).sum(dim=2)
        near = torch.where(good & (d2 <= R[j] ** 2), near, torch.full_like(near, math.inf))
        near, at = near.topk(min(40, near.shape[1]), dim=1, largest=False)
        j = j.gather(1, at)
        d = X[i][:, None, :] - X[j]
        q = d.norm(dim=2) / R[j]
        w = torch.where(q < 0.5, 1 - 6 * q * q * (1 - q), 2 * (1 - q) ** 3)
        w = torch.where((q < 1) & torch.isfinite(near), w, torch.zeros_like(w))
        basis = torch.cat([torch.ones_like(q)[:, :, None], d], dim=2)
        M = (w[:, :, None, None] * basis[:, :, :, None] * basis[:, :, None, :]).sum(dim=1)
        alone = torch.isfinite(near).sum(dim=1) == 1  # one neighbor, itself: value 1
        M = torch.where(alone[:, None, None], torch.eye(4, dtype=torch.float64, device=_dev()), M)
        scale = torch.tensor([1.0, 1 / p["h"], 1 / p["h"], 1 / p["h"]], dtype=torch.float64, device=_dev())
        e = torch.zeros(len(i), 4, 1, dtype=torch.float64, device=_dev())
        e[:, 0] = 1.0
        c = torch.linalg.solve(M * scale[:, None] * scale, e)[:, :, 0] * scale
        phi = w * (basis * c[:, None, :]).sum(dim=2)
        ids.append(j)
        vals.append(torch.where(alone[:, None], torch.isfinite(near).double(), phi))
    return torch.cat(ids), torch.cat(vals)


def _smoothed(case, p):
    """Reproducing-kernel runs: u = Phi d, cell force on u, f = Phi^T f_local."""
    nodal = case["kind"] == "nodal"
    nv = (case["nx"] + 1) * (case["ny"] + 1) * (case["nz"] + 1)
    ids, phi = _functions(p, case, nv)
    conn, ne = p["tconn"], len(p["tconn"])
    Xe = _corners(p["tX"], conn)
    B, V = _smoothed_hex(Xe) if nodal else next(_points(A.TET4, Xe))
    cell = conn[:, 0] if nodal else torch.arange(ne, device=_dev())
    ncell = nv if nodal else ne
    fold = lambda x: torch.zeros(ncell, dtype=torch.float64, device=_dev()).index_add_(0, cell, x)  # noqa: E731
    Vc = fold(V)
    st = dict(ep=torch.zeros(ncell, dtype=torch.float64, device=_dev()))

    def spread(x):
        return torch.zeros(len(p["tX"]), x.shape[1], dtype=torch.float64, device=_dev()).index_add_(
            0, ids.reshape(-1), (phi[:, :, None] * x[:, None, :]).reshape(-1, x.shape[1]))

    me = torch.zeros(len(p["tX"]), 1, dtype=torch.float64, device=_dev())
    for k in range(conn.shape[1]):
        me.index_add_(0, conn[:, k], (V * p["mat"]["rho"] / conn.shape[1])[:, None])
    m = spread(me)[:, 0]
    if nodal:
        p["free"] = p["free"] * (torch.arange(len(m), device=_dev()) < nv)[:, None]
        m = torch.where(m > 0, m, torch.ones_like(m))

    def force(d, inc, dt):
        u = (phi[:, :, None] * d[ids]).sum(dim=1)
        H = _grad(_corners(u, conn), B)
        if nodal and not case["f_bar"]:
            H = [[fold(H[i][j] * V) / Vc for j in range(3)] for i in range(3)]
        if nodal and case["f_bar"]:
            J = 1 + _jm1(H)
            Jb = (fold(J * V) / Vc)[cell]
            s = (Jb / J) ** (1.0 / 3.0)
            Hb = [[H[i][j] * s + (s - 1 if i == j else 0.0) for j in range(3)] for i in range(3)]
            Pb, new = _stress(p["kind"], Hb, p["lam"], p["mu"], p["mat"], st["ep"])
            F = _plus_i(H)
            pf = sum(Pb[i][j] * F[i][j] for i in range(3) for j in range(3))
            dual = (fold(s / (3 * Jb) * V * pf) / Vc)[cell]
            Fi = _inv(F)[0]
            P = [[Pb[i][j] * s + (dual - s / (3 * J) * pf) * J * Fi[j][i] for j in range(3)] for i in range(3)]
        else:
            P, new = _stress(p["kind"], H, p["lam"], p["mu"], p["mat"], st["ep"])
        Pe = [[P[i][j][cell] for j in range(3)] for i in range(3)] if nodal and not case["f_bar"] else P
        fl = torch.zeros_like(p["tX"])
        _scatter(fl, conn, B, Pe, V)
        if dt:
            st["ep"] = new
        return spread(fl), H, P

    out, got = _march(p, m, case["steps"], force, _t(p["v"]), p["dt"])
    if nodal:  # nodes without degrees of freedom keep their initial values
        inactive = torch.arange(len(m), device=_dev()) >= nv
        out["u"][inactive] = 0.0
        out["v"][inactive] = _t(p["v"])[inactive]
        out["a"][inactive] = 0.0
        out["f"][inactive] = 0.0
        return out
    out.update(H=_rows(got[1]), P=_rows(got[2]), state=st["ep"])
    return out


def _ensemble(case, seed):
    specs = _specimens(case, seed)
    X = np.concatenate([s["X"] for s in specs])
    first = np.cumsum([0] + [len(s["X"]) for s in specs])[:-1]
    per_e = [len(s["conn"]) for s in specs]
    lam, mu = zip(*(_lame(s["mat"]["E"], s["mat"]["nu"]) for s in specs))
    p = _on_device(dict(X=X, conn=np.concatenate([s["conn"] + n for s, n in zip(specs, first)]), fixed=None,
                        etype=A.HEX8, kind=MATERIALS[case["mat"]][0], mat=specs[0]["mat"]))
    p.update(lam=_t(np.repeat(lam, per_e)), mu=_t(np.repeat(mu, per_e)))
    dt = _t(np.repeat([s["dt"] for s in specs], [len(s["X"]) for s in specs]))[:, None]
    out, got = _march(p, _lumped(p), case["steps"], lambda u, inc, _: _force(p, u, None),
                      _t(np.concatenate([s["v"] for s in specs])), dt)
    out.update(H=_rows(got[1]), P=_rows(got[2]))
    return out


def _adjoint(case, seed, p):
    E, nu, target = (_t(x) for x in _parameter_fields(case, p, seed))
    p = _on_device(p)
    m = _lumped(p)
    leaves = [x.clone().requires_grad_(True) for x in (E, nu, _t(p["v"]))]
    dt = p["dt"]

    def accel(u, E, nu):
        q = dict(p)
        q["lam"], q["mu"] = _lame(E, nu)
        return _force(q, u, None)[0] / m[:, None]

    def step(u, v, a, E, nu):
        v = v + 0.5 * dt * a
        u = u + dt * v
        a = accel(u, E, nu)
        return u, v + 0.5 * dt * a, a

    again = functools.partial(torch.utils.checkpoint.checkpoint, use_reentrant=False)
    u, v = torch.zeros_like(leaves[2]), leaves[2]
    a = again(accel, u, leaves[0], leaves[1])
    for _ in range(case["steps"]):
        u, v, a = again(step, u, v, a, leaves[0], leaves[1])
    g = torch.autograd.grad(u, leaves, u.detach() - target)
    return dict(u=u.detach(), E_bar=g[0], nu_bar=g[1], v0_bar=g[2])


def _power(case, p):
    p = _on_device(p)
    m, l = _lumped(p)[:, None], _max_edge(p, len(p["X"]))[:, None]
    eps = 1e-5
    key = np.uint64(20261202) ^ np.arange(p["X"].size, dtype=np.uint64)
    with np.errstate(over="ignore"):  # splitmix64, the library's documented start vector
        key = key + np.uint64(0x9E3779B97F4A7C15)
        key = (key ^ (key >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        key = (key ^ (key >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    r = ((key ^ (key >> np.uint64(31))) >> np.uint64(11)).astype(np.float64) / 2.0 ** 53
    x = (2 * _t(r.reshape(-1, 3)) - 1) * (eps * l)
    u = torch.zeros_like(p["tX"])
    f0 = _force(p, u, None)[0]
    recent, dt, n, converged = [0.0] * 5, 1e-16, 50, False
    for k in range(50):
        last = dt
        x = (_force(p, u + x * l * eps, None)[0] - f0) / (l * eps * m)
        lam = float(x.norm())
        x = x / lam
        dt = recent[k % 5] = 2.0 / math.sqrt(lam)
        if abs(dt - last) < 1e-3 * dt or (k >= 5 and np.var(recent, ddof=1) < 1e-7 * np.mean(recent)):
            n, converged = k + 1, True
            break
    full = dt if converged else min(recent)
    out, got = _march(p, m[:, 0], case["steps"], lambda u, inc, _: _force(p, u, None), _t(p["v"]), 0.5 * full)
    out.update(H=_rows(got[1]), P=_rows(got[2]), increment=full, iterations=n, converged=converged)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        return _ensemble(case, seed)
    p = _problem(case, seed)
    if kind == "adjoint":
        return _adjoint(case, seed, p)
    if kind == "power":
        return _power(case, p)
    p = _on_device(p)
    if kind in ("rkpm", "nodal"):
        return _smoothed(case, p)
    if kind == "force":
        u = _t(_velocity(p["X"], seed, 100.0) * 30 * p["dt"])
        f, H, P, ep = _force(p, u, torch.zeros(len(p["conn"]), dtype=torch.float64, device=_dev()))
        return dict(f=f, H=_rows(H), P=_rows(P), **({"state": ep} if p["kind"] == A.J2 else {}))
    return _fem(case, p)
