"""Work that users of the dense BEM library have it do, as a list of timed cases.

Each case is one pass through the public API (`bempp_amd.api`): the weak form of one boundary
operator or of a single/double layer pair, the potential of a density, a frequency sweep, the
gradient of a loss with respect to the mesh, a GMRES solve. The meshes are closed spheres
(a subdivided icosahedron, 20 m^2 triangles, radially perturbed by the seed) and open curved
screens (2 m n triangles), from 80 triangles to the 20,480 of the benchmark.

`exact` restates every result in plain torch in 64 bits: the same quadrature rules (the 6-point
triangle rule for regular pairs, Sauter-Schwab points of order 4 for pairs sharing a vertex).
"""

import math
import os
import sys

import numpy as np
import torch

_PACKAGE = os.path.join(os.getcwd(), "bempp-cl_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: a coarse mesh while a script is written, or one panel of many; launches count
        {"name": "laplace_sl_p1_double_80", "path": "boundary", "op": "laplace_single_layer", "space": "P1",
         "mesh": "sphere", "m": 2, "n": 0, "k": 0.0, "ki": 0.0, "precision": "double"},
        # an electrostatics problem with piecewise constants, in the default precision
        {"name": "laplace_sl_dp0_double_1280", "path": "boundary", "op": "laplace_single_layer", "space": "DP0",
         "mesh": "sphere", "m": 8, "n": 0, "k": 0.0, "ki": 0.0, "precision": "double"},
        # acoustic scattering with a second-kind equation: the double layer in the default precision
        {"name": "helmholtz_dl_p1_double_3380", "path": "boundary", "op": "helmholtz_double_layer", "space": "P1",
         "mesh": "sphere", "m": 13, "n": 0, "k": 4.0, "ki": 0.0, "precision": "double"},
        # a sound-hard open screen in a lossy medium: hypersingular operator, complex wavenumber
        {"name": "helmholtz_hyp_p1_double_screen_4410", "path": "boundary", "op": "helmholtz_hypersingular",
         "space": "P1", "mesh": "screen", "m": 63, "n": 35, "k": 3.0, "ki": 0.4, "precision": "double"},
        # the benchmark's step: single and double layer of one space together, mixed precision, the largest mesh
        {"name": "helmholtz_sl_dl_p1_single_20480", "path": "pair", "op": "helmholtz_single_layer", "space": "P1",
         "mesh": "sphere", "m": 32, "n": 0, "k": 4.0, "ki": 0.0, "precision": "single"},
        # electromagnetic scattering in mixed precision, the benchmark's size
        {"name": "efie_rwg_single_5120", "path": "boundary", "op": "maxwell_electric_field", "space": "RWG",
         "mesh": "sphere", "m": 16, "n": 0, "k": 2.0, "ki": 0.0, "precision": "single"},
        # the same operator in the default precision on an ordinary, ragged mesh
        {"name": "efie_rwg_double_1620", "path": "boundary", "op": "maxwell_electric_field", "space": "RWG",
         "mesh": "sphere", "m": 9, "n": 0, "k": 3.0, "ki": 0.0, "precision": "double"},
        # the field of a solved density on a grid of observation points, mixed precision, the benchmark's size
        {"name": "helmholtz_sl_potential_single_20480_16384", "path": "potential", "op": "helmholtz_single_layer",
         "space": "P1", "mesh": "sphere", "m": 32, "n": 0, "k": 4.0, "ki": 0.0, "precision": "single",
         "points": 16384},
        # the electric field of a solved density in the default precision, odd sizes
        {"name": "efie_potential_double_1620_5003", "path": "potential", "op": "maxwell_electric_field",
         "space": "RWG", "mesh": "sphere", "m": 9, "n": 0, "k": 3.0, "ki": 0.0, "precision": "double",
         "points": 5003},
        # a frequency response: 32 wavenumbers of one mesh, mixed precision, the benchmark's size
        {"name": "sweep_dp0_single_5120_32", "path": "sweep", "op": "helmholtz_single_layer", "space": "DP0",
         "mesh": "sphere", "m": 16, "n": 0, "k": 16.0, "ki": 0.0, "precision": "single", "count": 32},
        # one step of shape optimisation: loss on boundary and field values, gradients of mesh and density
        {"name": "gradient_dp0_single_5120", "path": "gradient", "op": "helmholtz_single_layer", "space": "DP0",
         "mesh": "sphere", "m": 16, "n": 0, "k": 8.0, "ki": 0.0, "precision": "single", "points": 1024},
        # a first-kind equation solved by GMRES on the assembled operator, default precision
        {"name": "gmres_sl_p1_double_2000", "path": "solve", "op": "helmholtz_single_layer", "space": "P1",
         "mesh": "sphere", "m": 10, "n": 0, "k": 2.0, "ki": 0.0, "precision": "double"},
    ]


_SCALAR = ["laplace_single_layer", "laplace_double_layer", "laplace_adjoint_double_layer",
           "helmholtz_single_layer", "helmholtz_double_layer", "helmholtz_adjoint_double_layer"]


def _mesh(rng, low, high):
    """A sphere or a screen of about `low` to `high` triangles, log-uniform."""
    count = math.exp(rng.uniform(math.log(low), math.log(high)))
    if rng.random() < 0.6:
        return {"mesh": "sphere", "m": max(2, min(int(math.sqrt(high / 20)), round(math.sqrt(count / 20)))), "n": 0}
    m = max(4, round(math.sqrt(count / 2) * rng.uniform(0.7, 1.4)))
    return {"mesh": "screen", "m": m, "n": max(3, min(round(count / (2 * m)), high // (2 * m)))}


def _wavenumber(rng, op, mesh, damped=True):
    """Up to about eight elements a wavelength, sometimes in a lossy medium."""
    if op.startswith("laplace"):
        return {"k": 0.0, "ki": 0.0}
    elements = 20 * mesh["m"] ** 2 if mesh["mesh"] == "sphere" else 4 * mesh["m"] * mesh["n"]
    k = round(rng.uniform(0.1, 1.0) * 0.6 * math.sqrt(elements / 20), 3)
    return {"k": k, "ki": round(0.1 * k, 3) if damped and rng.random() < 0.25 else 0.0}


def draw(rng):
    path = rng.choice(["boundary"] * 6 + ["pair"] * 2 + ["potential"] * 3 + ["sweep", "gradient"])
    precision = rng.choice(["single", "double"])
    if path in ("boundary", "potential"):
        ops = _SCALAR[:2] + _SCALAR[3:5] if path == "potential" else _SCALAR + ["laplace_hypersingular",
                                                                                "helmholtz_hypersingular"]
        op = rng.choice(ops + ["maxwell_electric_field"] * 2 + ["maxwell_magnetic_field"])
        space = "RWG" if op.startswith("maxwell") else "P1" if "hyper" in op else rng.choice(["P1", "P1", "DP0", "DP1"])
        high = 8000 if precision == "single" else 4500
        mesh = _mesh(rng, 80, 3000 if space == "DP1" else high)
        case = {"path": path, "op": op, "space": space, **mesh, **_wavenumber(rng, op, mesh), "precision": precision}
        if path == "potential":
            case["points"] = round(math.exp(rng.uniform(math.log(60), math.log(20000))))
        return case
    if path == "pair":
        op = rng.choice(["laplace_single_layer", "helmholtz_single_layer"])
        mesh = _mesh(rng, 80, 16000 if precision == "single" else 6000)
        return {"path": path, "op": op, "space": rng.choice(["P1", "P1", "DP0"]), **mesh, **_wavenumber(rng, op, mesh),
                "precision": precision}
    op = "helmholtz_single_layer"
    if path == "sweep":
        mesh = _mesh(rng, 80, 5000 if precision == "single" else 1300)
        return {"path": path, "op": op, "space": "DP0", **mesh, **_wavenumber(rng, op, mesh, False),
                "precision": precision, "count": rng.randint(2, 40 if precision == "single" else 12)}
    mesh = _mesh(rng, 80, 6000 if precision == "single" else 3000)
    return {"path": path, "op": op, "space": "DP0", **mesh, **_wavenumber(rng, op, mesh, False),
            "precision": precision, "points": rng.randint(60, 3000)}


def work(case):
    """Outputs written and inputs read once; FLOP of one evaluation of every element pair's 36 point
    pairs (each unordered pair once where the matrix is symmetric): distance 8, its root and
    reciprocal 2, e^{ikr} 4, a normal derivative 8, and the sums over shape functions."""
    F = _elements_of(case)
    rows = {"DP0": F, "DP1": 3 * F, "P1": F // 2 + 2, "RWG": 3 * F // 2}[case["space"]]
    value = (8 if case["precision"] == "single" else 16) // (2 if case["op"].startswith("laplace") else 1)
    parts = 1 if case["op"].startswith("laplace") else 2
    layer = 10 + (6 if parts == 2 else 0)
    shape = {"DP0": 0, "DP1": 6, "P1": 6, "RWG": 8}[case["space"]] * parts + 2 * parts
    normal = 8 if "double" in case["op"] or "magnetic" in case["op"] else 0
    mesh = 24 * (F // 2 + 2) + 12 * F
    if case["path"] == "potential":
        kd = 3 if case["op"].startswith("maxwell") else 1
        return {"bytes": mesh + 16 * rows + 24 * case["points"] + 2 * value * kd * case["points"],
                "flops": 6.0 * F * case["points"] * (layer + normal + 8 * kd)}
    if case["path"] == "solve":
        return {"bytes": 30.0 * rows * rows * value, "flops": 30.0 * 8 * rows * rows}
    pairs = 36.0 * F * F
    if case["path"] == "sweep":
        return {"bytes": mesh + float(value) * rows * rows * case["count"],
                "flops": pairs / 2 * (10 + 8 * case["count"])}
    if case["path"] == "gradient":
        return {"bytes": mesh + 32.0 * rows + 24 * case["points"] + float(value) * rows * rows,
                "flops": pairs / 2 * (layer + shape) + pairs * 26}
    if case["path"] == "pair":
        return {"bytes": mesh + 2.0 * value * rows * rows, "flops": pairs / 2 * (layer + 16 + 3 * shape)}
    symmetric = "single" in case["op"] or "hyper" in case["op"] or "electric" in case["op"]
    return {"bytes": mesh + float(value) * rows * rows,
            "flops": pairs * (0.5 if symmetric else 1.0) * (layer + normal + shape)}


def tolerance(case):
    """Relative errors of another correct implementation at the same precision (see `exact`)."""
    if case["path"] == "solve":
        return {"rel": 1e-10, "max": 1e-8}  # the same iterates: rounding times the condition of the basis
    if case["precision"] == "double":
        return {"rel": 2e-12, "max": 1e-10} if case["path"] == "gradient" else {"rel": 1e-13, "max": 1e-11}
    return {"rel": 1e-6, "max": 1e-4}


# ------------------------------------------------------------------ meshes and inputs
_PHI = (1.0 + 5.0**0.5) / 2.0


def _sphere(m):
    """Icosahedron with every edge cut into m parts, on the unit sphere: (vertices (V, 3), triangles (F, 3))."""
    corners = np.array([[-1, _PHI, 0], [1, _PHI, 0], [-1, -_PHI, 0], [1, -_PHI, 0], [0, -1, _PHI], [0, 1, _PHI],
                        [0, -1, -_PHI], [0, 1, -_PHI], [_PHI, 0, -1], [_PHI, 0, 1], [-_PHI, 0, -1], [-_PHI, 0, 1]])
    faces = [(0, 11, 5), (0, 5, 1), (0, 1, 7), (0, 7, 10), (0, 10, 11), (1, 5, 9), (5, 11, 4), (11, 10, 2),
             (10, 7, 6), (7, 1, 8), (3, 9, 4), (3, 4, 2), (3, 2, 6), (3, 6, 8), (3, 8, 9), (4, 9, 5), (2, 4, 11),
             (6, 2, 10), (8, 6, 7), (9, 8, 1)]
    ij = np.array([(i, j) for i in range(m + 1) for j in range(m + 1 - i)])
    at = {(i, j): n for n, (i, j) in enumerate(ij.tolist())}
    local = []
    for i in range(m):
        for j in range(m - i):
            local.append((at[i, j], at[i + 1, j], at[i, j + 1]))
            if i + j < m - 1:
                local.append((at[i + 1, j], at[i + 1, j + 1], at[i, j + 1]))
    points = np.concatenate([corners[a] + (ij[:, :1] * (corners[b] - corners[a]) + ij[:, 1:] * (corners[c] - corners[a])) / m
                             for a, b, c in faces])
    triangles = np.concatenate([np.array(local) + n * len(ij) for n in range(20)])
    _, first, inverse = np.unique(np.round(points, 9), axis=0, return_index=True, return_inverse=True)
    points = points[first]
    return points / np.linalg.norm(points, axis=1)[:, None], inverse.ravel()[triangles]


def _screen(m, n):
    """A screen of m x n squares, each cut in two, 2 wide."""
    x, y = np.meshgrid(np.arange(m + 1), np.arange(n + 1), indexing="ij")
    points = np.stack([2.0 * x.ravel() / m - 1.0, (2.0 * y.ravel() - n) / m, np.zeros(x.size)], axis=1)
    a = (np.arange(m)[:, None] * (n + 1) + np.arange(n)[None, :]).ravel()
    low = np.stack([a, a + n + 1, a + n + 2], axis=1)
    high = np.stack([a, a + n + 2, a + 1], axis=1)
    return points, np.stack([low, high], axis=1).reshape(-1, 3)


def _elements_of(case):
    return 20 * case["m"] ** 2 if case["mesh"] == "sphere" else 2 * case["m"] * case["n"]


def _geometry(case, seed):
    """Vertices (V, 3) and triangles (F, 3): the seed bends the surface by a few per cent."""
    rng = np.random.default_rng([seed, 1])
    v, t = _sphere(case["m"]) if case["mesh"] == "sphere" else _screen(case["m"], case["n"])
    waves, phases = rng.uniform(-2.0, 2.0, (6, 3)), rng.uniform(0.0, 2.0 * np.pi, 6)
    bend = 0.02 * np.cos(v @ waves.T + phases).sum(axis=1)
    if case["mesh"] == "sphere":
        return v * (1.0 + bend)[:, None], t
    return v + np.stack([np.zeros(len(v)), np.zeros(len(v)), 2.0 * bend], axis=1), t


def _dof_count(case, v, t):
    return {"DP0": len(t), "DP1": 3 * len(t)}.get(case["space"]) or int(_dof_map(case["space"], v, t)[0].max()) + 1


def _density(case, seed, n):
    rng = np.random.default_rng([seed, 2])
    c = rng.standard_normal(n)
    return c if case["op"].startswith("laplace") else c + 1j * rng.standard_normal(n)


def _points(case, seed):
    """Observation points 1.5 to 3 from the centre."""
    rng = np.random.default_rng([seed, 3])
    p = rng.standard_normal((case["points"], 3))
    return p / np.linalg.norm(p, axis=1)[:, None] * rng.uniform(1.5, 3.0, (case["points"], 1))


def _wavenumbers(case):
    return np.linspace(case["k"] / case["count"], case["k"], case["count"])


def _k(case):
    return complex(case["k"], case["ki"]) if case["ki"] else case["k"]


def _operator(case, state, op=None):
    import bempp_amd.api as bempp

    family, _, name = (op or case["op"]).partition("_")
    options = () if family == "laplace" else (_k(case),)
    make = getattr(getattr(bempp.operators.boundary, family), name)
    return make(state["domain"], state["domain"], state["dual"], *options, precision=case["precision"])


def prepare(case, seed):
    import bempp_amd.api as bempp

    v, t = _geometry(case, seed)
    grid = bempp.Grid(np.ascontiguousarray(v.T), np.ascontiguousarray(t.T))
    state = {"case": case, "grid": grid}
    if case["path"] == "gradient":
        from bempp_amd.api.differentiable import SingleLayerProblem

        dev = torch.device("cuda")
        state["problem"] = SingleLayerProblem(grid.elements, case["k"], precision=case["precision"])
        state["vertices"] = torch.from_numpy(v).to(dev)
        state["density"] = torch.from_numpy(_density(case, seed, len(t))).to(dev)
        state["target"] = torch.from_numpy(_density(case, seed + 7919, len(t))).to(dev)
        state["points"] = torch.from_numpy(_points(case, seed)).to(dev)
        return state
    kind, degree = {"DP0": ("DP", 0), "DP1": ("DP", 1), "P1": ("P", 1), "RWG": ("RWG", 0)}[case["space"]]
    state["domain"] = bempp.function_space(grid, kind, degree)
    state["dual"] = bempp.function_space(grid, "SNC", 0) if kind == "RWG" else state["domain"]
    if case["path"] == "potential":
        family, _, name = case["op"].partition("_")
        options = () if family == "laplace" else (_k(case),)
        make = getattr(getattr(bempp.operators.potential, family), name)
        state["potential"] = make(state["domain"], np.ascontiguousarray(_points(case, seed).T), *options,
                                  precision=case["precision"])
        state["density"] = bempp.GridFunction(
            state["domain"], coefficients=_density(case, seed, state["domain"].global_dof_count))
    if case["path"] == "solve":
        state["operator"] = _operator(case, state)
        state["operator"].weak_form()
        b = _density(case, seed, state["domain"].global_dof_count)
        state["rhs"] = bempp.GridFunction(state["domain"], projections=b, dual_space=state["dual"])
    return state


def run(state):
    import bempp_amd.api as bempp

    case = state["case"]
    if case["path"] == "boundary":
        return _operator(case, state).weak_form().tensor
    if case["path"] == "pair":
        from bempp_amd.api.assembly.boundary_operator import assemble_weak_forms

        ops = [_operator(case, state), _operator(case, state, case["op"].replace("single", "double"))]
        return [form.tensor for form in assemble_weak_forms(ops)]
    if case["path"] == "potential":
        return state["potential"].evaluate(state["density"])
    if case["path"] == "sweep":
        forms = bempp.operators.boundary.helmholtz.single_layer_frequency_sweep(
            state["domain"], state["domain"], state["dual"], _wavenumbers(case), precision=case["precision"])
        return [form.tensor for form in forms]
    if case["path"] == "solve":
        solution, info = bempp.linalg.gmres(state["operator"], state["rhs"], tol=1e-5)
        return solution.coefficients, info
    from bempp_amd.api.differentiable import single_layer_apply, single_layer_potential

    v = state["vertices"].clone().requires_grad_(True)
    c = state["density"].clone().requires_grad_(True)
    y = single_layer_apply(v, c, state["problem"])
    u = single_layer_potential(v, c, state["points"], state["problem"])
    loss = (y - state["target"]).abs().pow(2).sum() + u.abs().pow(2).sum()
    loss.backward()
    return {"values": y.detach(), "field": u.detach(), "vertices": v.grad, "density": c.grad}


# ------------------------------------------------------------------ 64-bit restatement
def _triangle_rule():
    """The symmetric 6-point rule of degree 4 on the reference triangle: points (6, 2), weights (6,)."""
    points, weights = [], []
    for b, w in ((0.44594849091596488632, 0.22338158967801146570), (0.091576213509770743460, 0.10995174365532186764)):
        a = 1.0 - 2.0 * b
        points += [(b, b), (a, b), (b, a)]
        weights += [0.5 * w] * 3
    return np.array(points), np.array(weights)


def _singular_rule(shared):
    """Sauter-Schwab points (test (N, 2), trial (N, 2)) and weights for triangles that coincide (3
    shared vertices) or share the edge 0-1 (2) or the vertex 0 (1), from 4-point Gauss rules."""
    x, w = np.polynomial.legendre.leggauss(4)
    x, w = 0.5 * (x + 1.0), 0.5 * w
    s, a, b, c = (g.ravel() for g in np.meshgrid(x, x, x, x, indexing="ij"))
    weight = np.einsum("i,j,k,l->ijkl", w, w, w, w).ravel() * s**3
    one = np.ones_like(s)
    if shared == 3:
        weight = weight * a**2 * b
        maps = [(one, 1 - a + a * b, 1 - a * b * c, 1 - a), (one, a - a * b + a * b * c, 1 - a * b, a - a * b),
                (1 - a * b * c, a - a * b * c, one, a - a * b)]
        maps = [(m, one) for m in maps] + [(m[2:] + m[:2], one) for m in maps]
    elif shared == 2:
        weight = weight * a**2
        maps = [((one, a * c, 1 - a * b, a - a * b), one), ((one, a, 1 - a * b * c, a * b - a * b * c), b),
                ((1 - a * b, a - a * b, one, a * b * c), b), ((1 - a * b * c, a * b - a * b * c, one, a), b),
                ((1 - a * b * c, a - a * b * c, one, a * b), b)]
    else:
        weight = weight * b
        maps = [((one, a, b, b * c), one), ((b, b * c, one, a), one)]
    # the maps' triangle has the corners (0, 0), (1, 0), (1, 1)
    test = np.concatenate([np.stack([s * (m[0] - m[1]), s * m[1]], axis=1) for m, _ in maps])
    trial = np.concatenate([np.stack([s * (m[2] - m[3]), s * m[3]], axis=1) for m, _ in maps])
    return test, trial, np.concatenate([weight * f for _, f in maps])


def _dof_map(space, v, t):
    """(dofs (F, shapes), multipliers): P1 dofs are the vertices off the boundary, RWG dofs the inner
    edges in the order they first occur, positive on the neighbour of lower index."""
    F = len(t)
    if space in ("DP0", "DP1"):
        s = 1 if space == "DP0" else 3
        return np.arange(s * F).reshape(F, s), np.ones((F, s))
    edges = np.sort(t[:, [[0, 1], [2, 0], [1, 2]]], axis=2).reshape(-1, 2)
    _, first, inverse, count = np.unique(edges[:, 0] * (len(v) + 1) + edges[:, 1], return_index=True,
                                         return_inverse=True, return_counts=True)
    inverse = inverse.ravel()
    if space == "P1":
        inner = np.ones(len(v), bool)
        inner[edges[first[count == 1]].ravel()] = False
        number = np.cumsum(inner) - 1
        return np.where(inner[t], number[t], 0), inner[t].astype(float)
    rank = np.full(len(first), -1)
    used = np.flatnonzero(count == 2)
    rank[used[np.argsort(first[used])]] = np.arange(len(used))
    dofs = rank[inverse].reshape(F, 3)
    owner = (first // 3)[inverse].reshape(F, 3) == np.arange(F)[:, None]
    return np.where(dofs < 0, 0, dofs), np.where(dofs < 0, 0.0, np.where(owner, 1.0, -1.0))


class _Surface:
    """Triangles on the GPU in 64 bits; differentiable in the vertices."""

    def __init__(self, case, vertices, t):
        dev = vertices.device
        self.t = torch.from_numpy(t).to(dev)
        self.space = case["space"]
        corners = vertices[self.t]  # (F, 3, 3)
        self.v0, self.e1, self.e2 = corners[:, 0], corners[:, 1] - corners[:, 0], corners[:, 2] - corners[:, 0]
        cross = torch.linalg.cross(self.e1, self.e2)
        self.J = torch.linalg.vector_norm(cross, dim=1)
        self.n = cross / self.J[:, None]
        dofs, mult = _dof_map(case["space"], vertices.detach().cpu().numpy(), t)
        self.dofs, self.mult = torch.from_numpy(dofs).to(dev), torch.from_numpy(mult).to(dev)
        self.ndof = int(self.dofs.max()) + 1
        self.lengths = torch.stack([torch.linalg.vector_norm(e, dim=1) for e in (self.e1, self.e2, self.e1 - self.e2)], 1)

    def at(self, e, x):
        """Points of the triangles e (E,) at reference points x (E or 1, N, 2): (E, N, 3)."""
        return self.v0[e, None] + self.e1[e, None] * x[..., :1] + self.e2[e, None] * x[..., 1:]

    def basis(self, kind, e, x):
        """Components of a shape function field times the multipliers, each (E, N, shapes)."""
        m = self.mult[e][:, None]
        if kind in ("phi", "n phi"):
            u, w = x[..., 0], x[..., 1]
            phi = torch.ones_like(u)[..., None] if self.space == "DP0" else torch.stack([1 - u - w, u, w], -1)
            phi = phi * m
            return [phi] if kind == "phi" else [phi * self.n[e][:, None, None, d] for d in range(3)]
        if kind == "curl":  # n x grad phi
            c = torch.stack([self.e1[e] - self.e2[e], self.e2[e], -self.e1[e]], 1) / self.J[e][:, None, None]
            return [(m * c[:, None, :, d]).expand(-1, x.shape[1], -1) for d in range(3)]
        scale = m * (self.lengths / self.J[:, None])[e][:, None]
        if kind == "div":
            return [(2.0 * scale).expand(-1, x.shape[1], -1)]
        o = torch.tensor([[0.0, 1.0], [1.0, 0.0], [0.0, 0.0]], dtype=x.dtype, device=x.device)
        r = x[..., None, :] - o  # the RWG function vanishes at the vertex o
        return [scale * (self.e1[e][:, None, None, d] * r[..., 0] + self.e2[e][:, None, None, d] * r[..., 1])
                for d in range(3)]


def _terms(case, k, op):
    """The operator as a list of (test field, trial field, factor, kernel) whose products are summed
    over the fields' components; the kernel is a name for _kernel."""
    if op.endswith("hypersingular"):
        return [("curl", "curl", 1.0, "G"), ("n phi", "n phi", -k * k, "G")][: 1 if k == 0 else 2]
    if op == "maxwell_electric_field":
        return [("rwg", "rwg", -1j * k, "G"), ("div", "div", -1.0 / (1j * k), "G")]
    return [("phi", "phi", 1.0, op.partition("_")[2])]


def _kernel(name, k, d, nx, ny):
    """Kernel values for d = y - x (three components)."""
    r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
    r = torch.sqrt(r2)
    real = k == 0
    G = 1.0 / (4.0 * math.pi * r)
    if not real:
        G = torch.polar(G * torch.exp(-k.imag * r) if k.imag else G, k.real * r)
    if name in ("G", "single_layer"):
        return G
    g = -G / r2 if real else G * torch.complex(-1.0 - k.imag * r, k.real * r) / r2
    if name == "gradient":
        return g
    if name == "double_layer":
        return g * (d[0] * ny[0] + d[1] * ny[1] + d[2] * ny[2])
    return -g * (d[0] * nx[0] + d[1] * nx[1] + d[2] * nx[2])


_PERMUTED = [((1, 2), 0, 1.0), ((2, 1), 0, -1.0), ((2, 0), 1, 1.0), ((0, 2), 1, -1.0), ((0, 1), 2, 1.0), ((1, 0), 2, -1.0)]


def _blocks(case, k, op, S, e, f, x, y, contract):
    """Sum of the operator's terms; contract(test field, kernel, trial field) sums over the points."""
    X, Y = S.at(e, x), S.at(f, y)
    total = 0.0
    if op == "maxwell_magnetic_field":  # gradient kernel times (x - y) . (test x trial)
        d, K = contract.kernel("gradient", k, X, Y, S.n[e], S.n[f])
        A, B = S.basis("rwg", e, x), S.basis("rwg", f, y)
        for (a, b), c, sign in _PERMUTED:
            total = total - sign * contract(A[a], K * d[c], B[b])
        return total
    for test, trial, factor, name in _terms(case, k, op):
        _, K = contract.kernel(name, k, X, Y, S.n[e], S.n[f])
        for A, B in zip(S.basis(test, e, x), S.basis(trial, f, y)):
            total = total + factor * contract(A, K, B)
    return total


class _Regular:
    """Test points x all trial points: (E, P, i), (E P, F Q), (F, Q, j) -> (E, i, F, j)."""

    def __init__(self, weights, Je, Jf, skip):
        self.w, self.Je, self.Jf, self.skip = weights, Je, Jf, skip

    def kernel(self, name, k, X, Y, nx, ny):
        E, P, F, Q = X.shape[0], X.shape[1], Y.shape[0], Y.shape[1]
        d = [(Y[..., c].reshape(1, -1) - X[..., c].reshape(-1, 1)) for c in range(3)]
        close = self.skip[:, None, :, None].expand(E, P, F, Q).reshape(E * P, F * Q)
        d[0] = torch.where(close, torch.ones((), dtype=X.dtype, device=X.device), d[0])
        nx = [nx[:, None, c].expand(E, P).reshape(-1, 1) for c in range(3)]
        ny = [ny[:, None, c].expand(F, Q).reshape(1, -1) for c in range(3)]
        K = _kernel(name, k, d, nx, ny)
        return d, torch.where(close, torch.zeros((), dtype=K.dtype, device=X.device), K)

    def __call__(self, A, K, B):
        (E, P, i), (F, Q, j) = A.shape, B.shape
        B = (B * self.w[:, None] * self.Jf[:, None, None]).to(K.dtype)
        A = (A * self.w[:, None] * self.Je[:, None, None]).to(K.dtype)
        K = K.view(E * P, F, Q)
        T = sum(K[:, :, q, None] * B[:, q] for q in range(Q)) if Q > 1 else K * B
        T = T.reshape(E, P, F * j)
        return sum(A[:, p, :, None] * T[:, p, None, :] for p in range(P)).view(E, i, F, j)


class _Singular:
    """Pairs with points of their own: (n, N, i), (n, N), (n, N, j) -> (n, i, j)."""

    def __init__(self, weights, J):
        self.w = weights[None] * J[:, None]

    def kernel(self, name, k, X, Y, nx, ny):
        d = [Y[..., c] - X[..., c] for c in range(3)]
        return d, _kernel(name, k, d, [nx[:, None, c] for c in range(3)], [ny[:, None, c] for c in range(3)])

    def __call__(self, A, K, B):
        K = K * self.w
        return torch.stack([(A[..., i, None] * K[..., None] * B).sum(1) for i in range(A.shape[-1])], 1)


def _neighbours(t):
    """Ordered pairs of triangles sharing vertices: (e, f, vertices of e, vertices of f) by the number
    shared; for an edge the pair of vertices is in the order in which it stands in f."""
    F, V = len(t), int(t.max()) + 1
    from_vertex = [[] for _ in range(V)]
    for e, corners in enumerate(t.tolist()):
        for v in corners:
            from_vertex[v].append(e)
    found = {1: [], 2: [], 3: []}
    corners = t.tolist()
    for e in range(F):
        for f in sorted({f for v in corners[e] for f in from_vertex[v]}):
            shared = [(i, j) for j, w in enumerate(corners[f]) for i, v in enumerate(corners[e]) if v == w]
            found[len(shared)].append((e, f, [i for i, _ in shared], [j for _, j in shared]))
    return found


def _moved(points, vertices):
    """Rule points whose shared vertex is 0 (edge 0-1) on triangles that share the given vertices."""
    if len(vertices) == 3:
        return points
    bary = np.concatenate([1.0 - points.sum(axis=1, keepdims=True), points], axis=1)
    if len(vertices) == 1:
        order = [0, 1, 2]
        order[0], order[vertices[0]] = order[vertices[0]], order[0]
    else:
        order = list(vertices) + [3 - sum(vertices)]
    new = np.empty_like(bary)
    new[:, order] = bary
    return new[:, 1:]


def _singular_pairs(case, S, t):
    """(e, f, test points, trial points, weights) groups of the pairs sharing a vertex."""
    groups = []
    for shared, pairs in _neighbours(t).items():
        test, trial, weights = _singular_rule(shared)
        kinds = {}
        for e, f, i, j in pairs:
            kinds.setdefault((tuple(i), tuple(j)) if shared < 3 else ((0, 1, 2), (0, 1, 2)), []).append((e, f))
        for (i, j), members in kinds.items():
            ef = torch.tensor(members, device=S.J.device)
            put = [torch.from_numpy(_moved(p, s)).to(S.J.device)[None] for p, s in ((test, i), (trial, j))]
            groups.append((ef[:, 0], ef[:, 1], *put, torch.from_numpy(weights).to(S.J.device)))
    return groups


def _chunks(count, size):
    return [(a, min(a + size, count)) for a in range(0, count, size)]


def _rule_on(dev):
    points, weights = _triangle_rule()
    return torch.from_numpy(points).to(dev)[None], torch.from_numpy(weights).to(dev)


def _matrix(case, k, op, S, t):
    """The dense Galerkin matrix in 64 bits."""
    dev = S.J.device
    k = complex(k) if k else 0
    out = torch.zeros((S.ndof, S.ndof), dtype=torch.complex128 if k else torch.float64, device=dev)
    x, w = _rule_on(dev)
    F = len(S.t)
    every = torch.arange(F, device=dev)
    flat = S.dofs.reshape(-1)
    for a, b in _chunks(F, max(1, 25_000_000 // (36 * F))):
        e = every[a:b]
        skip = (S.t[e][:, :, None, None] == S.t.T[None, None]).any(1).any(1)
        V = _blocks(case, k, op, S, e, every, x, x, _Regular(w, S.J[e], S.J, skip))
        E, i = V.shape[:2]
        rows = torch.zeros((E * i, S.ndof), dtype=V.dtype, device=dev)
        rows.index_add_(1, flat, V.reshape(E * i, -1))
        out.index_add_(0, S.dofs[e].reshape(-1), rows)
    for e, f, p, q, weights in _singular_pairs(case, S, t):
        for a, b in _chunks(len(e), max(1, 4_000_000 // len(weights))):
            V = _blocks(case, k, op, S, e[a:b], f[a:b], p, q, _Singular(weights, S.J[e[a:b]] * S.J[f[a:b]]))
            out.index_put_((S.dofs[e[a:b]][:, :, None].expand_as(V), S.dofs[f[a:b]][:, None].expand_as(V)), V, True)
    return out


def _field(case, k, op, S, coefficients, points):
    """Potential values (components, points) in 64 bits."""
    dev = S.J.device
    k = complex(k) if k else 0
    x, w = _rule_on(dev)
    every = torch.arange(len(S.t), device=dev)
    Y = S.at(every, x).reshape(-1, 3)
    scale = w[None, :] * S.J[:, None]
    local = coefficients[S.dofs][:, None]

    def source(kind):
        return [((c * local).sum(-1) * scale).reshape(-1) for c in S.basis(kind, every, x)]

    normals = S.n[:, None].expand(-1, 6, 3).reshape(-1, 3)
    maxwell = op.startswith("maxwell")
    current = source("rwg") if maxwell else source("phi")
    charge = source("div")[0] if maxwell else None
    values = []
    for a, b in _chunks(len(points), max(1, 20_000_000 // len(Y))):
        X = points[a:b]
        d = [Y[None, :, c] - X[:, None, c] for c in range(3)]
        if not maxwell:
            K = _kernel(op.partition("_")[2], k, d, None, [normals[None, :, c] for c in range(3)])
            values.append((K.to(torch.complex128) @ current[0].to(torch.complex128))[None])
            continue
        g = _kernel("gradient", k, d, None, None)
        if op == "maxwell_electric_field":
            G = _kernel("G", k, d, None, None)
            # grad_x G = (y - x) (1 - ikr) G / r^2 = -(y - x) g, times charge / (ik)
            values.append(torch.stack([1j * k * (G @ current[c]) + ((g * d[c]) @ charge) / (1j * k) for c in range(3)]))
        else:
            turn = [[(g * -d[c]) @ current[j] for j in range(3)] for c in range(3)]
            values.append(torch.stack([turn[(c + 1) % 3][(c + 2) % 3] - turn[(c + 2) % 3][(c + 1) % 3] for c in range(3)]))
    return torch.cat(values, 1)


def _gradient(case, seed, v, t, dev):
    vertices = torch.from_numpy(v).to(dev).requires_grad_(True)
    c = torch.from_numpy(_density(case, seed, len(t))).to(dev).requires_grad_(True)
    target = torch.from_numpy(_density(case, seed + 7919, len(t))).to(dev)
    points = torch.from_numpy(_points(case, seed)).to(dev)
    k, op, F = complex(case["k"]), case["op"], len(t)
    groups = _singular_pairs(case, _Surface(case, vertices.detach(), t), t)
    y = torch.empty(F, dtype=torch.complex128, device=dev)
    u = []
    for a, b in _chunks(F, max(1, 8_000_000 // (36 * F))):
        S = _Surface(case, vertices, t)
        x, w = _rule_on(dev)
        every = torch.arange(F, device=dev)
        e = every[a:b]
        skip = (S.t[e][:, :, None, None] == S.t.T[None, None]).any(1).any(1)
        V = _blocks(case, k, op, S, e, every, x, x, _Regular(w, S.J[e], S.J, skip))
        rows = V.reshape(b - a, F) @ c
        for e, f, p, q, weights in groups:
            own = (e >= a) & (e < b)
            if own.any():
                e, f = e[own], f[own]
                V = _blocks(case, k, op, S, e, f, p, q, _Singular(weights, S.J[e] * S.J[f]))
                rows = rows.index_add(0, e - a, V.reshape(-1) * c[f])
        (rows - target[a:b]).abs().pow(2).sum().backward()
        y[a:b] = rows.detach()
    for a, b in _chunks(len(points), max(1, 8_000_000 // (6 * F))):
        part = _field(case, k, op, _Surface(case, vertices, t), c, points[a:b])[0]
        part.abs().pow(2).sum().backward()
        u.append(part.detach())
    return {"values": y, "field": torch.cat(u), "vertices": vertices.grad, "density": c.grad}


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    v, t = _geometry(case, seed)
    if case["path"] == "gradient":
        return _gradient(case, seed, v, t, dev)
    S = _Surface(case, torch.from_numpy(v).to(dev), t)
    k, op = _k(case), case["op"]
    if case["path"] == "boundary":
        return _matrix(case, k, op, S, t)
    if case["path"] == "pair":
        return [_matrix(case, k, name, S, t) for name in (op, op.replace("single", "double"))]
    if case["path"] == "potential":
        points = torch.from_numpy(_points(case, seed)).to(dev)
        density = torch.from_numpy(_density(case, seed, S.ndof).astype(complex)).to(dev)
        values = _field(case, k, op, S, density, points)
        return values.real if op.startswith("laplace") else values
    if case["path"] == "sweep":
        return [_matrix(case, float(q), op, S, t) for q in _wavenumbers(case)]
    b = torch.from_numpy(_density(case, seed, S.ndof)).to(dev)
    return torch.linalg.solve(_matrix(case, k, op, S, t), b).cpu().numpy(), None
