"""The assembly work that a user of this framework has it do, as cases to time.

A case is one pass through the public entry points of `cudolfinx` on data
that is already on the GPU: a system A + b (matrix, right-hand side, lifting,
Dirichlet values), a batch of systems, a Newton step, or one product with an
assembled matrix.  Mesh, spaces, forms and matrix handles are what a program
keeps between assemblies; coefficients, states and boundary values change from
pass to pass and come from the seed.  Helmholtz problems have no coefficient:
their mesh geometry comes from the seed, with everything built on it.

`exact` evaluates the same discrete systems with plain torch in float64, from
the mesh and dofmap arrays alone.
"""
from __future__ import annotations

import itertools
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "cuda-dolfinx_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)


# --------------------------------------------------------------------- cases
def listed():
    return [
        # the smallest systems (unit tests, coarse grids of a hierarchy): launches and host calls
        {"name": "poisson_p1_7", "family": "poisson", "degree": 1, "n": 7},
        # large scalar problem of the lowest order: little arithmetic per byte
        {"name": "poisson_p1_50", "family": "poisson", "degree": 1, "n": 50},
        # ordinary scalar problem, odd size
        {"name": "poisson_p2_25", "family": "poisson", "degree": 2, "n": 25},
        # high order scalar problem
        {"name": "poisson_p3_24", "family": "poisson", "degree": 3, "n": 24},
        # small structural model, odd size
        {"name": "elasticity_p2_13", "family": "elasticity", "n": 13},
        # the largest: a structural model of 2.7 million dofs
        {"name": "elasticity_p2_48", "family": "elasticity", "n": 48},
        # high order wave problem on curved hexahedra driven from its boundary, double precision
        {"name": "helmholtz_q3_24_f64", "family": "helmholtz", "n": 24, "precision": 64,
         "boundary_data": True},
        # the same operator with single precision element arithmetic, zero on the boundary
        {"name": "helmholtz_q3_24_f32", "family": "helmholtz", "n": 24, "precision": 32,
         "boundary_data": False},
        # many small independent meshes in one launch, element tensors of
        # degree 2 and 3 in single precision
        {"name": "batch_48_f32", "family": "batch", "instances": 48, "nmin": 4, "nmax": 16,
         "sizes_seed": 3, "precision": 32},
        # reassembly of a discontinuous Galerkin Newton step (Jacobian, residual, energy)
        {"name": "newton_dg1_32", "family": "newton", "degree": 1, "n": 32},
        # nonlinear problem given by its element kernels alone: Jacobian and residual
        {"name": "nonlinear_p2_20", "family": "nonlinear", "degree": 2, "n": 20},
        # the product a Krylov solver takes with the assembled matrix
        {"name": "product_elasticity_32", "family": "product", "n": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["poisson", "poisson", "elasticity", "elasticity", "helmholtz", "batch",
                         "newton", "nonlinear", "product"])
    if family == "poisson":
        degree = rng.choice([1, 2, 3])
        return {"family": family, "degree": degree,
                "n": _log_int(rng, 4, {1: 50, 2: 36, 3: 24}[degree])}
    if family == "elasticity":
        return {"family": family, "n": _log_int(rng, 4, 40)}
    if family == "helmholtz":
        return {"family": family, "n": _log_int(rng, 4, 24), "precision": rng.choice([64, 64, 32, 16]),
                "boundary_data": rng.random() < 0.5}
    if family == "batch":
        return {"family": family, "instances": _log_int(rng, 4, 64), "nmin": 4,
                "nmax": rng.randint(5, 16), "sizes_seed": rng.randrange(1000),
                "precision": rng.choice([64, 32])}
    if family == "newton":
        degree = rng.choice([1, 1, 2])
        return {"family": family, "degree": degree, "n": _log_int(rng, 4, {1: 32, 2: 14}[degree])}
    if family == "nonlinear":
        degree = rng.choice([1, 2])
        return {"family": family, "degree": degree, "n": _log_int(rng, 4, {1: 32, 2: 20}[degree])}
    return {"family": family, "n": _log_int(rng, 6, 32)}


# ------------------------------------------------------------ kept by a program
_kept = {}          # the last discretisation: {"key": ..., "D": ...}


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k != "name"))


def _discretisation(case, on_device=True):
    """Mesh, spaces and forms of a case (and, on_device, compiled forms and
    matrices): what a program lays out once and keeps."""
    key = (_key(case), on_device)
    if _kept.get("key") != key:
        _kept.clear()
        D = _BUILD[case["family"]](case)
        if on_device:
            _to_device(case, D)
        _kept.update(key=key, D=D)
    return _kept["D"]


def _boundary_nodes(V, axis=None):
    from mifem.fem import locate_dofs_topological
    mesh = V.mesh
    f = mesh.exterior_facets if axis is None else mesh.locate_boundary_facets(
        lambda x: np.isclose(x[axis], 0.0))
    return locate_dofs_topological(V, 2, f)


def _build_poisson(case):
    from mifem import forms
    from mifem.fem import Function, functionspace
    from mifem.mesh import create_unit_cube
    mesh = create_unit_cube(case["n"])
    V = functionspace(mesh, ("P", case["degree"]))
    V1 = V if case["degree"] == 1 else functionspace(mesh, ("P", 1))
    kappa, f = Function(functionspace(mesh, ("DG", 0)), "kappa"), Function(V1, "f")
    return {"V": V, "V1": V1, "mesh": mesh, "a": forms.stiffness(V, kappa), "L": forms.source(V, f),
            "nodes": _boundary_nodes(V)}


def _build_elasticity(case):
    from mifem import forms
    from mifem.fem import Constant, Function, functionspace
    from mifem.mesh import create_unit_cube
    mesh = create_unit_cube(case["n"])
    V = functionspace(mesh, ("P", 2), shape=(3,))
    D0 = functionspace(mesh, ("DG", 0))
    right = mesh.locate_boundary_facets(lambda x: np.isclose(x[0], 1.0))
    load = Constant([0.0, 0.0, -1.0])
    L = forms.linear_sum(forms.source(V, load), forms.facet_source(V, load, right))
    return {"V": V, "mesh": mesh, "a": forms.elasticity(V, Function(D0, "mu"), Function(D0, "lambda")),
            "L": L, "right": right, "nodes": _boundary_nodes(V, axis=0)}


def _build_helmholtz(case, seed=0):
    from mifem import problems
    P = problems.helmholtz_q3(case["n"], seed=seed)
    return {"V": P.V, "mesh": P.mesh, "a": P.a, "L": P.L, "nodes": _boundary_nodes(P.V)}


def _build_batch(case):
    from mifem import batch
    B = batch.many_poisson(case["instances"], seed=case["sizes_seed"], nmin=case["nmin"], nmax=case["nmax"])
    return {"groups": B.groups}


def _build_newton(case):
    from mifem import problems
    from mifem.dgforms import sipg_energy
    P = problems.dg_plaplace(case["n"], degree=case["degree"])
    return {"V": P.V, "mesh": P.mesh, "J": P.a, "F": P.L, "E": sipg_energy(P.V, P.extras["u"])}


def _build_nonlinear(case):
    from mifem.mesh import create_unit_cube
    from mifem.nonlinear import reference_test_forms
    mesh = create_unit_cube(case["n"], jitter=0.2, seed=7)
    R = reference_test_forms(mesh, case["degree"])
    return {"V": R["u"].function_space, "mesh": mesh, "a": R["matrix"][0], "L": R["vector"][0],
            "nodes": R["bcs"][0].dofs}


_BUILD = {"poisson": _build_poisson, "elasticity": _build_elasticity, "helmholtz": _build_helmholtz,
          "batch": _build_batch, "newton": _build_newton, "nonlinear": _build_nonlinear,
          "product": _build_elasticity}


def _to_device(case, D):
    import cudolfinx as cufem
    asm = D["asm"] = cufem.CUDAAssembler()
    options = {"precision": case["precision"]} if case.get("precision", 64) != 64 else None
    if case["family"] == "batch":
        D["a"] = [cufem.form(g.a, options=options if g.degree >= 2 else None) for g in D["groups"]]
        D["L"] = [cufem.form(g.L) for g in D["groups"]]
        D["A"] = [asm.create_matrix(a) for a in D["a"]]
        D["matrices"], D["vectors"] = cufem.CUDABatch(D["a"]), cufem.CUDABatch(D["L"])
    elif case["family"] == "newton":
        D["J"], D["F"], D["E"] = (cufem.form(D[k]) for k in "JFE")
        D["A"] = asm.create_matrix(D["J"])
        D["system"] = cufem.CUDASystem(D["J"], D["F"], D["E"])
    else:
        D["a"], D["L"] = cufem.form(D["a"], options=options), cufem.form(D["L"])
        D["A"] = asm.create_matrix(D["a"])


# --------------------------------------------------------------------- inputs
def _normal(seed, field, *shape):
    g = torch.Generator(device="cuda")
    g.manual_seed(1009 * int(seed) + field)
    return torch.randn(*shape, generator=g, dtype=torch.float64, device="cuda")


def _uniform(seed, field, *shape):
    g = torch.Generator(device="cuda")
    g.manual_seed(1009 * int(seed) + field)
    return torch.rand(*shape, generator=g, dtype=torch.float64, device="cuda")


def _boundary_values(seed, nodes, bs, zero=False):
    """Values of the constrained dofs, in the order of the nodes."""
    if zero:
        return np.zeros((len(nodes), bs))
    return 0.1 * np.random.default_rng([int(seed), 5]).standard_normal((len(nodes), bs))


def _bc(V, nodes, values):
    from mifem.fem import Function, dirichletbc
    g = Function(V, "g")
    g.x.reshape(-1, V.bs)[nodes] = values
    return dirichletbc(g, nodes, V)


def _state_values(V, seed, noise):
    """A smooth field with a little noise: a Newton iterate."""
    x = torch.as_tensor(V.node_coordinates, device="cuda")
    smooth = torch.sin(math.pi * x[:, 0]) * torch.sin(math.pi * x[:, 1]) * torch.cos(x[:, 2])
    return (smooth + noise * _normal(seed, 3, V.num_nodes)).contiguous()


def _coefficients(case, D, seed):
    """Values of the bilinear and the linear form's coefficients, in their order."""
    family = case["family"]
    nc = D["mesh"].num_cells if "mesh" in D else 0
    if family == "poisson":
        return [torch.exp(_normal(seed, 1, nc))], [_normal(seed, 2, D["V1"].num_nodes)]
    if family in ("elasticity", "product"):
        return [1.0 + 9.0 * _uniform(seed, k, nc) for k in (1, 2)], []
    if family == "nonlinear":
        u = _state_values(D["V"], seed, 0.05)
        kappa = 1.0 + 0.5 * _uniform(seed, 2, D["V"].num_nodes)
        return [u, kappa], [u, kappa]
    return [], []


class _View:
    """Device memory of the framework, for torch.as_tensor."""

    def __init__(self, address, n):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f8", "data": (address, False),
                                         "version": 3}


def _values(A):
    return torch.as_tensor(_View(A.device_arrays()[2], A.nnz), device="cuda")


def _vector(b):
    return torch.as_tensor(_View(b.data.address, b.size), device="cuda")


def prepare(case, seed):
    family = case["family"]
    if family == "helmholtz":
        D = _build_helmholtz(case, seed)
        _kept.clear()
        _to_device(case, D)
    else:
        D = _discretisation(case)
    asm = D["asm"]
    s = {"family": family, "D": D, "asm": asm}
    if family == "batch":
        s["kappa"] = [torch.exp(_normal(seed, 10 + k, g.mesh.num_cells)) for k, g in enumerate(D["groups"])]
        s["b"] = [asm.create_vector(L) for L in D["L"]]
        s["bcs"] = []
        for k, g in enumerate(D["groups"]):
            nodes = g.bcs[0].dofs
            s["bcs"].append(asm.pack_bcs([_bc(g.V, nodes, _boundary_values(seed + k, nodes, 1))]))
        s["out"] = [{"A": _values(A), "b": _vector(b)} for A, b in zip(D["A"], s["b"])]
    elif family == "newton":
        s["u"] = _state_values(D["V"], seed, 0.01)
        s["b"], s["e"] = asm.create_vector(D["F"]), torch.zeros(1, dtype=torch.float64, device="cuda")
        s["out"] = {"J": _values(D["A"]), "F": _vector(s["b"]), "E": s["e"]}
    elif family == "product":
        # the matrix stays, the vector changes from product to product
        if "assembled" not in D:
            D["coefficients"] = _coefficients(case, D, 0)[0]
            D["bcs"] = asm.pack_bcs([_bc(D["V"], D["nodes"], 0.0)])
            for j, c in enumerate(D["coefficients"]):
                D["a"].set_coefficient_device(j, c.data_ptr(), c.numel())
            asm.assemble_matrix(D["a"], D["A"], bcs=D["bcs"])
            D["assembled"] = True
        s["x"] = _normal(seed, 4, D["A"].ncols)
        s["y"] = torch.empty(D["A"].nrows, dtype=torch.float64, device="cuda")
    else:
        s["ca"], s["cL"] = _coefficients(case, D, seed)
        s["b"] = asm.create_vector(D["L"])
        zero = not case.get("boundary_data", True)
        s["bcs"] = asm.pack_bcs([_bc(D["V"], D["nodes"],
                                     _boundary_values(seed, D["nodes"], D["V"].bs, zero))])
        if family == "nonlinear":
            s["x0"] = asm.create_vector(D["L"])
            _vector(s["x0"]).copy_(s["ca"][0])
        s["out"] = {"A": _values(D["A"]), "b": _vector(s["b"])}
    torch.cuda.synchronize()
    return s


# ----------------------------------------------------------------------- pass
def _bind(form, coefficients):
    for j, c in enumerate(coefficients):
        form.set_coefficient_device(j, c.data_ptr(), c.numel())


def run(state):
    s, D, asm = state, state["D"], state["asm"]
    if s["family"] == "product":
        return D["A"].mult(s["x"], s["y"])
    if s["family"] == "newton":
        for k in "JFE":
            _bind(D[k], [s["u"]])
        D["system"].assemble(asm, D["A"], s["b"], value=s["e"])
        return s["out"]
    if s["family"] == "batch":
        for a, kappa in zip(D["a"], s["kappa"]):
            _bind(a, [kappa])
        D["matrices"].assemble(asm, D["A"], s["bcs"])
        D["vectors"].assemble_vectors(asm, s["b"])
        for a, b, bcs in zip(D["a"], s["b"], s["bcs"]):
            asm.apply_lifting(b, [a], [bcs])
        D["vectors"].set_bc(asm, s["b"], s["bcs"])
        return s["out"]
    _bind(D["a"], s["ca"])
    _bind(D["L"], s["cL"])
    asm.assemble_matrix(D["a"], D["A"], bcs=s["bcs"])
    asm.assemble_vector(D["L"], s["b"])
    if s["family"] == "nonlinear":
        # Newton's right-hand side: the update moves the iterate x0 onto the boundary values
        asm.apply_lifting(s["b"], [D["a"]], [s["bcs"]], x0=[s["x0"]], scale=-1.0)
        asm.set_bc(s["b"], s["bcs"], D["V"], x0=s["x0"], scale=-1.0)
    else:
        asm.apply_lifting(s["b"], [D["a"]], [s["bcs"]])
        asm.set_bc(s["b"], s["bcs"], D["V"])
    return s["out"]


# ----------------------------------------------------------------------- work
def _tet_counts(n):
    """Vertices, edges, faces and cells of n^3 cubes of 6 tetrahedra."""
    return ((n + 1) ** 3, 3 * n * (n + 1) ** 2 + 3 * n * n * (n + 1) + n ** 3, 12 * n ** 3 + 6 * n * n, 6 * n ** 3)


def _tet_pairs(n, k):
    """Pairs of P_k nodes that share a tetrahedron: over all simplices, the
    pairs whose supports together are that simplex."""
    def full(d):
        return sum((-1) ** (d - j) * math.comb(d + 1, j + 1) * math.comb(k + j, j) ** 2 for j in range(d + 1))
    return sum(c * full(d) for d, c in enumerate(_tet_counts(n)))


def _tet_work(n, k, bs, coefficients, nq):
    """Values and b written, the block pattern, geometry, dofmap and coefficients read."""
    nc, nodes, pairs, nd = 6 * n ** 3, (k * n + 1) ** 3, _tet_pairs(n, k), math.comb(k + 3, 3)
    return {"bytes": 8 * bs * bs * pairs + 4 * pairs + 4 * (nodes + 1) + 8 * bs * nodes
            + 24 * (n + 1) ** 3 + 16 * nc + 4 * nd * nc + 8 * coefficients * nc,
            "flops": nc * nd * nd * (12 + 18 * (bs > 1) * nq)}


def _work_add(ws):
    ws = list(ws)
    return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}


def work(case):
    family, n = case["family"], case.get("n")
    if family == "poisson":
        return _tet_work(n, case["degree"], 1, 2, 1)
    if family == "elasticity":
        return _tet_work(n, 2, 3, 2, 4)
    if family == "nonlinear":
        k = case["degree"]
        w = _tet_work(n, k, 1, 2, 1)
        # u and kappa at the nodes, (k + 2)^3 points of exp(u) and gradients
        w["flops"] = 6 * n ** 3 * (k + 2) ** 3 * (8 * math.comb(k + 3, 3) ** 2)
        return w
    if family == "helmholtz":
        nodes, nnz = (3 * n + 1) ** 3, (16 * n - (n - 1)) ** 3
        # sum-factorised element matrices: about 3 k multiply-adds per row of 64
        return {"bytes": 12 * nnz + 8 * nodes + 4 * (nodes + 1) + 24 * (n + 1) ** 3 + 4 * 72 * n ** 3,
                "flops": n ** 3 * 64 * 2 * 3000}
    if family == "batch":
        rng = np.random.default_rng(case["sizes_seed"])
        sizes = rng.integers(case["nmin"], case["nmax"] + 1, size=case["instances"])
        degrees = rng.choice(np.asarray((1, 2, 3)), size=case["instances"])
        return _work_add(_tet_work(int(m), int(k), 1, 1, 1) for m, k in zip(sizes, degrees))
    if family == "newton":
        nd, nc, nint = math.comb(case["degree"] + 3, 3), 6 * n ** 3, 12 * n ** 3 - 6 * n * n
        return {"bytes": 8 * nd * nd * (nc + 2 * nint) + 8 * nd * nc + 8 * nd * nc + 24 * (n + 1) ** 3
                + 16 * nc + 16 * nint, "flops": nint * (case["degree"] + 1) ** 2 * 8 * (2 * nd) ** 2}
    pairs, nodes = _tet_pairs(n, 2), (2 * n + 1) ** 3
    return {"bytes": 12 * 9 * pairs + 2 * 24 * nodes + 12 * nodes, "flops": 2 * 9 * pairs}


# ---------------------------------------------------------------------- exact
def _gauss_jacobi(m, alpha):
    """Nodes and weights on [0, 1] for the weight (1 - t)^alpha (Golub-Welsch)."""
    i = np.arange(m, dtype=np.float64)
    s = 2 * i + alpha
    diag = np.where(s * (s + 2) == 0, -alpha / (alpha + 2), -alpha * alpha / np.where(s * (s + 2) == 0, 1, s * (s + 2)))
    j = np.arange(1, m, dtype=np.float64)
    t = 2 * j + alpha
    off = np.sqrt(4 * j * (j + alpha) * j * (j + alpha) / (t * t * (t + 1) * (t - 1)))
    x, v = np.linalg.eigh(np.diag(diag) + np.diag(off, 1) + np.diag(off, -1))
    return (x + 1) / 2, v[0] ** 2 / (alpha + 1)


def _simplex_rule(dim, m):
    """Collapsed Gauss-Jacobi rule with m points per direction."""
    rules = [_gauss_jacobi(m, float(a)) for a in range(dim - 1, -1, -1)]
    pts, w = [], []
    for ids in itertools.product(range(m), repeat=dim):
        rest, p, weight = 1.0, [], 1.0
        for (x, wx), i in zip(rules, ids):
            p.append(x[i] * rest)
            rest *= 1.0 - x[i]
            weight *= wx[i]
        pts.append(p)
        w.append(weight)
    return np.array(pts), np.array(w)


_EDGES = [(2, 3), (1, 3), (1, 2), (0, 3), (0, 2), (0, 1)]
_FACES = [(1, 2, 3), (0, 2, 3), (0, 1, 3), (0, 1, 2)]


def _tet_nodes(k):
    """Barycentric indices of the P_k nodes: vertices, edges, faces."""
    out = [[k * (a == v) for a in range(4)] for v in range(4)]
    for a, b in _EDGES:
        for s in range(1, k):
            out.append([k - s if v == a else s if v == b else 0 for v in range(4)])
    for f in _FACES:
        for t in range(1, k):
            for s in range(1, k - t):
                m = [0, 0, 0, 0]
                m[f[0]], m[f[1]], m[f[2]] = k - s - t, s, t
                out.append(m)
    return np.array(out, dtype=np.float64)


def _tet_basis(k, pts):
    """(values (nq, nd), reference gradients (nq, nd, 3)) of P_k at points, on the GPU."""
    mons = [e for e in itertools.product(range(k + 1), repeat=3) if sum(e) <= k]

    def monomials(X, d=None):
        cols = []
        for e in mons:
            p = list(e)
            c = 1.0
            if d is not None:
                c, p[d] = float(p[d]), max(p[d] - 1, 0)
            cols.append(c * X[:, 0] ** p[0] * X[:, 1] ** p[1] * X[:, 2] ** p[2])
        return np.stack(cols, axis=1)

    C = np.linalg.inv(monomials(_tet_nodes(k)[:, 1:] / k))
    val = monomials(pts) @ C
    grad = np.stack([monomials(pts, d) @ C for d in range(3)], axis=-1)
    return torch.as_tensor(val, device="cuda"), torch.as_tensor(grad, device="cuda")


def _dev(a, dtype=None):
    t = torch.as_tensor(np.ascontiguousarray(a), device="cuda")
    return t if dtype is None else t.to(dtype)


def _affine(x, cells):
    """K[c][r][d] = dX_r / dx_d and |det J| of affine tetrahedra."""
    p = x[cells]
    J = (p[:, 1:] - p[:, :1]).transpose(1, 2)          # J[d][r] = dx_d / dX_r
    return torch.linalg.inv(J), torch.linalg.det(J).abs()


class _Pattern:
    """The block CSR of pairs of nodes that share an entity, and sums into it."""

    def __init__(self, rows, cols, nb, bs):
        """rows, cols: (entities, m) node numbers; every pair of an entity couples."""
        self.nb, self.bs = nb, bs
        keys = (rows[:, :, None] * nb + cols[:, None, :]).reshape(-1)
        self.keys, self.at = torch.unique(keys, return_inverse=True)
        self.at = self.at.view(rows.shape[0], -1)
        self.v = torch.zeros(self.keys.numel(), bs, bs, dtype=torch.float64, device="cuda")

    def add(self, e, A):
        """A: (chunk, m, bs, m, bs) element matrices of the entities e."""
        self.v.index_add_(0, self.at[e].reshape(-1),
                          A.permute(0, 1, 3, 2, 4).reshape(-1, self.bs, self.bs))

    def values(self, constrained=None):
        """CSR values, the rows and columns of constrained dofs replaced by the identity's."""
        R, C = self.keys // self.nb, self.keys % self.nb
        v, bs = self.v, self.bs
        if constrained is not None:
            free = (~constrained).view(self.nb, bs).to(torch.float64)
            v = v * free[R][:, :, None] * free[C][:, None, :]
            on = torch.nonzero(R == C).flatten()
            v[on] += torch.diag_embed(1.0 - free[R[on]])
        count = torch.bincount(R, minlength=self.nb)
        start = torch.cumsum(count, 0) - count
        k = torch.arange(bs, device="cuda")
        pos = (bs * bs * start[R] + bs * (torch.arange(R.numel(), device="cuda") - start[R]))[:, None, None] \
            + (bs * count[R])[:, None, None] * k[None, :, None] + k[None, None, :]
        out = torch.empty(v.numel(), dtype=torch.float64, device="cuda")
        out[pos.reshape(-1)] = v.reshape(-1)
        return out


def _chunks(n, size):
    return (slice(i, min(i + size, n)) for i in range(0, n, size))


def _second_order(mesh, dofmap, nb, k, block, source, constrained, g, bs, x0=None, scale=1.0, size=20000):
    """A and b of a form on affine tetrahedra: block(e, G) gives element
    matrices from G_ij[p][q] = int d_p phi_i d_q phi_j (or from the cells e
    alone), source(e) element vectors."""
    x, cells, dm = _dev(mesh.x), _dev(mesh.cells, torch.int64), _dev(dofmap, torch.int64)
    P = _Pattern(dm, dm, nb, bs)
    b = torch.zeros(nb, bs, dtype=torch.float64, device="cuda")
    pts, w = _simplex_rule(3, max(1, k))
    _, dphi = _tet_basis(k, pts)
    R = torch.einsum("q,qir,qjs->ijrs", torch.as_tensor(w, device="cuda"), dphi, dphi)
    lift = (g - (x0 if x0 is not None else 0.0)) * constrained
    for e in _chunks(cells.shape[0], size):
        K, det = _affine(x, cells[e])
        A = block(e, K, det, R)
        P.add(e, A)
        be = source(e, K, det) - scale * torch.einsum("ciajb,cjb->cia", A, lift.view(nb, bs)[dm[e]])
        b.index_add_(0, dm[e].reshape(-1), be.reshape(-1, bs))
    b = b.reshape(-1)
    return P, torch.where(constrained, scale * (g - (x0 if x0 is not None else 0.0)), b)


def _constraint(nodes, values, nb, bs):
    mask = torch.zeros(nb, bs, dtype=torch.bool, device="cuda")
    g = torch.zeros(nb, bs, dtype=torch.float64, device="cuda")
    at = _dev(nodes, torch.int64)
    mask[at] = True
    g[at] = _dev(values)
    return mask.reshape(-1), g.reshape(-1)


def _exact_poisson(mesh, V, k, kappa, f, dof1, nodes, values):
    phi, _ = _tet_basis(k, (r := _simplex_rule(3, k + 1))[0])
    psi, _ = _tet_basis(1, r[0])
    M = torch.einsum("q,qi,qk->ik", torch.as_tensor(r[1], device="cuda"), phi, psi)
    d1 = _dev(dof1, torch.int64)
    on, g = _constraint(nodes, values, V.num_nodes, 1)

    def block(e, K, det, R):
        G = torch.einsum("crd,csd->crs", K, K) * (det * kappa[e])[:, None, None]
        return torch.einsum("crs,ijrs->cij", G, R)[:, :, None, :, None]

    P, b = _second_order(mesh, V.dofmap, V.num_nodes, k, block,
                         lambda e, K, det: (det[:, None] * (f[d1[e]] @ M.T))[:, :, None], on, g, 1)
    return {"A": P.values(on), "b": b}


def _exact_elasticity(D, mu, lam, nodes, values):
    V, mesh = D["V"], D["mesh"]
    phi, _ = _tet_basis(2, (r := _simplex_rule(3, 2))[0])
    load = torch.tensor([0.0, 0.0, -1.0], dtype=torch.float64, device="cuda")
    m = torch.einsum("q,qi->i", torch.as_tensor(r[1], device="cuda"), phi)
    on, g = _constraint(nodes, values, V.num_nodes, 3)
    eye = torch.eye(3, dtype=torch.float64, device="cuda")

    def block(e, K, det, R):
        G = torch.einsum("crp,ijrs,csq->cijpq", K, R, K) * det[:, None, None, None, None]
        tr = torch.einsum("cijpp->cij", G)
        B = mu[e][:, None, None, None, None] * (tr[..., None, None] * eye + G.transpose(3, 4)) \
            + lam[e][:, None, None, None, None] * G
        return B.permute(0, 1, 3, 2, 4)

    P, b = _second_order(mesh, V.dofmap, V.num_nodes, 2, block,
                         lambda e, K, det: det[:, None, None] * m[None, :, None] * load, on, g, 3)
    # traction on x = 1
    q2, w2 = _simplex_rule(2, 2)
    b = b.view(-1, 3)
    x, cells, dm = _dev(mesh.x), _dev(mesh.cells, torch.int64), _dev(V.dofmap, torch.int64)
    right = _dev(D["right"], torch.int64)
    for lf, f in enumerate(_FACES):
        c = right[right[:, 1] == lf, 0]
        if c.numel() == 0:
            continue
        p = x[cells[c][:, list(f)]]
        area = torch.linalg.norm(torch.linalg.cross(p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]), dim=1)
        ph, _ = _tet_basis(2, _facet_points(lf, q2))
        m2 = torch.einsum("q,qi->i", torch.as_tensor(w2, device="cuda"), ph)
        b.index_add_(0, dm[c].reshape(-1), (area[:, None, None] * m2[None, :, None] * load).reshape(-1, 3))
    return P, torch.where(on, g, b.reshape(-1)), on


def _facet_points(lf, q2):
    X = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]], dtype=np.float64)
    lam = np.stack([1 - q2[:, 0] - q2[:, 1], q2[:, 0], q2[:, 1]], axis=1)
    return lam @ X[list(_FACES[lf])]


def _exact_nonlinear(D, k, u, kappa, nodes, values):
    V = D["V"]
    pts, w = _simplex_rule(3, k + 2)
    phi, dphi = _tet_basis(k, pts)
    w = torch.as_tensor(w, device="cuda")
    S = torch.einsum("q,qir,qjs->ijrs", w, dphi, dphi)
    dm = _dev(V.dofmap, torch.int64)
    on, g = _constraint(nodes, values, V.num_nodes, 1)

    def weight(e, det):
        return w * torch.exp(u[dm[e]] @ phi.T) * (kappa[dm[e]] @ phi.T) * det[:, None]

    def stiffness(K, det):
        G = torch.einsum("crd,csd->crs", K, K) * det[:, None, None]
        return torch.einsum("crs,ijrs->cij", G, S)

    def block(e, K, det, R):
        A = torch.einsum("cq,qi,qj->cij", weight(e, det), phi, phi) + stiffness(K, det)
        return A[:, :, None, :, None]

    def source(e, K, det):
        return (weight(e, det) @ phi + torch.einsum("cij,cj->ci", stiffness(K, det), u[dm[e]]))[:, :, None]

    P, b = _second_order(D["mesh"], V.dofmap, V.num_nodes, k, block, source, on, g, 1, x0=u, scale=-1.0)
    return {"A": P.values(on), "b": b}


def _exact_helmholtz(D, nodes, values, k2=25.0):
    V, mesh = D["V"], D["mesh"]
    t, w1 = _gauss_jacobi(4, 0.0)
    r = 1.0 / math.sqrt(5.0)
    node = np.array([0.0, (1 - r) / 2, (1 + r) / 2, 1.0])
    C = np.linalg.inv(np.vander(node, 4, increasing=True))
    L = np.vander(t, 4, increasing=True) @ C
    G = np.stack([0 * t, 1 + 0 * t, 2 * t, 3 * t * t], axis=1) @ C

    def tensor(fx, fy, fz):          # (q, i), x fastest in both
        return np.einsum("ai,bj,ck->cbakji", fx, fy, fz).reshape(fx.shape[0] ** 3, -1)
    phi = _dev(tensor(L, L, L))
    B = torch.stack([_dev(tensor(G, L, L)), _dev(tensor(L, G, L)), _dev(tensor(L, L, G))], dim=-1)
    l1 = np.stack([1 - t, t], axis=1)
    d1 = np.stack([-1 + 0 * t, 1 + 0 * t], axis=1)
    dpsi = torch.stack([_dev(tensor(d1, l1, l1)), _dev(tensor(l1, d1, l1)), _dev(tensor(l1, l1, d1))], dim=-1)
    w = _dev(np.einsum("a,b,c->cba", w1, w1, w1).reshape(-1))
    x, cells, dm = _dev(mesh.x), _dev(mesh.cells, torch.int64), _dev(V.dofmap, torch.int64)
    nb = V.num_nodes
    on, g = _constraint(nodes, values, nb, 1)
    P = _Pattern(dm, dm, nb, 1)
    b = torch.zeros(nb, dtype=torch.float64, device="cuda")
    for e in _chunks(cells.shape[0], 500):
        J = torch.einsum("cvd,qvr->cqdr", x[cells[e]], dpsi)
        det = torch.linalg.det(J).abs() * w
        K = torch.linalg.inv(J)
        M = torch.einsum("cqrd,cqsd->cqrs", K, K) * det[..., None, None]
        F = torch.einsum("cqrs,qjs->cqrj", M, B)
        A = torch.einsum("qir,cqrj->cij", B, F) - k2 * torch.einsum("cq,qi,qj->cij", det, phi, phi)
        P.add(e, A[:, :, None, :, None])
        be = det @ phi - torch.einsum("cij,cj->ci", A, (g * on)[dm[e]])
        b.index_add_(0, dm[e].reshape(-1), be.reshape(-1))
    return {"A": P.values(on), "b": torch.where(on, g, b)}


def _exact_newton(D, k, u, p=3.0, eps=1e-3, alpha=2.0, f=1.0):
    V, mesh = D["V"], D["mesh"]
    x, cells, nc, nd = _dev(mesh.x), _dev(mesh.cells, torch.int64), mesh.num_cells, V.element.ndofs
    inter, ext = _dev(mesh.interior_facets, torch.int64), _dev(mesh.exterior_facets, torch.int64)
    me = torch.arange(nc, device="cuda")[:, None]
    both = torch.stack([inter[:, 0], inter[:, 2]], dim=1)
    # couplings of a cell with itself, of the two cells of a facet
    keys = torch.cat([(me * nc + me).reshape(-1), (both[:, :, None] * nc + both[:, None, :]).reshape(-1)])
    P = object.__new__(_Pattern)
    P.nb, P.bs = nc, nd
    P.keys = torch.unique(keys)
    P.v = torch.zeros(P.keys.numel(), nd, nd, dtype=torch.float64, device="cuda")

    def add(r, c, A):
        P.v.index_add_(0, torch.searchsorted(P.keys, r * nc + c), A)

    F, E = torch.zeros(nc, nd, dtype=torch.float64, device="cuda"), 0.0
    u = u.view(nc, nd)
    K, det = _affine(x, cells)
    pts, w = _simplex_rule(3, max(1, k))
    phi, dphi = _tet_basis(k, pts)
    w = torch.as_tensor(w, device="cuda")
    for e in _chunks(nc, 20000):
        gr = torch.einsum("qir,crd->cqid", dphi, K[e])
        gu = torch.einsum("cqid,ci->cqd", gr, u[e])
        s2 = eps * eps + (gu * gu).sum(-1)
        mu, dmu, fw = 1.0 + s2 ** ((p - 2) / 2), (p - 2) * s2 ** ((p - 4) / 2), w * det[e][:, None]
        gi = torch.einsum("cqid,cqd->cqi", gr, gu)
        add(me[e, 0], me[e, 0], torch.einsum("cq,cqid,cqjd->cij", fw * mu, gr, gr)
            + torch.einsum("cq,cqi,cqj->cij", fw * dmu, gi, gi))
        F[e] += torch.einsum("cq,cqi->ci", fw * mu, gi) - f * torch.einsum("cq,qi->ci", fw, phi)
        E += float((fw * (s2 ** (p / 2) / p + 0.5 * (gu * gu).sum(-1) - f * (u[e] @ phi.T))).sum())
    q2, w2 = _simplex_rule(2, k + 1)
    w2 = torch.as_tensor(w2, device="cuda")
    tab = [_tet_basis(k, _facet_points(lf, q2)) for lf in range(4)]
    fphi, fgrad = torch.stack([t[0] for t in tab]), torch.stack([t[1] for t in tab])
    faces = torch.tensor(_FACES, device="cuda")
    edge = x[cells]
    h = torch.stack([torch.linalg.norm(edge[:, a] - edge[:, b], dim=1)
                     for a, b in itertools.combinations(range(4), 2)]).max(0).values

    def normal(c, lf):
        q = edge[c]
        at = faces[lf]
        v = torch.gather(q, 1, at[:, :, None].expand(-1, -1, 3))
        nrm = torch.linalg.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
        ds = torch.linalg.norm(nrm, dim=1)
        away = q[torch.arange(len(c), device="cuda"), lf] - v[:, 0]
        nrm = nrm / ds[:, None]
        return torch.where(((nrm * away).sum(1) > 0)[:, None], -nrm, nrm), ds

    c, lf = ext[:, 0], ext[:, 1]
    _, ds = normal(c, lf)
    ph = fphi[lf]
    fw, uq = w2 * ds[:, None] * alpha, torch.einsum("fqi,fi->fq", fphi[lf], u[c])
    add(c, c, torch.einsum("fq,fqi,fqj->fij", fw, ph, ph))
    F.index_add_(0, c, torch.einsum("fq,fqi->fi", fw * uq, ph))
    E += float((0.5 * fw * uq * uq).sum())
    for e in _chunks(inter.shape[0], 40000):
        c0, l0, c1, l1 = inter[e].T
        n, ds = normal(c0, l0)
        sig = 30.0 * k * k / (0.5 * (h[c0] + h[c1]))
        jump = torch.cat([fphi[l0], -fphi[l1]], dim=2)
        dn = 0.5 * torch.cat([torch.einsum("fqir,frd,fd->fqi", fgrad[lf], K[c], n)
                              for c, lf in ((c0, l0), (c1, l1))], dim=2)
        fw, uu = w2 * ds[:, None], torch.cat([u[c0], u[c1]], dim=1)
        A = -torch.einsum("fq,fqi,fqj->fij", fw, jump, dn)
        A = A + A.transpose(1, 2) + torch.einsum("fq,fqi,fqj->fij", fw * sig[:, None], jump, jump)
        ju, du = torch.einsum("fqi,fi->fq", jump, uu), torch.einsum("fqi,fi->fq", dn, uu)
        v = torch.einsum("fq,fqi->fi", fw * (sig[:, None] * ju - du), jump) - torch.einsum("fq,fqi->fi", fw * ju, dn)
        for a, ca in enumerate((c0, c1)):
            F.index_add_(0, ca, v[:, a * nd:(a + 1) * nd])
            for b, cb in enumerate((c0, c1)):
                add(ca, cb, A[:, a * nd:(a + 1) * nd, b * nd:(b + 1) * nd])
        E += float((fw * (0.5 * sig[:, None] * ju * ju - du * ju)).sum())
    return {"J": P.values(), "F": F.reshape(-1), "E": torch.tensor([E], dtype=torch.float64)}


def exact(case, seed):
    family = case["family"]
    if family == "helmholtz":
        D = _build_helmholtz(case, seed)
        zero = not case["boundary_data"]
        return _exact_helmholtz(D, D["nodes"], _boundary_values(seed, D["nodes"], 1, zero))
    D = _discretisation(case, on_device=False)
    if family == "batch":
        out = []
        for k, g in enumerate(D["groups"]):
            nodes, dof1 = g.bcs[0].dofs, g.mesh.cells
            one = torch.ones(g.mesh.num_vertices, dtype=torch.float64, device="cuda")
            out.append(_exact_poisson(g.mesh, g.V, g.degree, torch.exp(_normal(seed, 10 + k, g.mesh.num_cells)),
                                      one, dof1, nodes, _boundary_values(seed + k, nodes, 1)))
        return out
    if family == "newton":
        return _exact_newton(D, case["degree"], _state_values(D["V"], seed, 0.01))
    if family == "product":
        mu, lam = _coefficients(case, D, 0)[0]
        P, _, on = _exact_elasticity(D, mu, lam, D["nodes"], np.zeros((len(D["nodes"]), 3)))
        free = (~on).to(torch.float64).view(-1, 3)
        x = _normal(seed, 4, D["V"].size).view(-1, 3)
        R, C = P.keys // P.nb, P.keys % P.nb
        y = torch.zeros_like(x).index_add_(0, R, torch.einsum("eab,eb->ea", P.v, (x * free)[C]))
        return (y * free + x * (1.0 - free)).reshape(-1)
    values = _boundary_values(seed, D["nodes"], D["V"].bs)
    ca, cL = _coefficients(case, D, seed)
    if family == "poisson":
        return _exact_poisson(D["mesh"], D["V"], case["degree"], ca[0], cL[0], D["V1"].dofmap, D["nodes"], values)
    if family == "nonlinear":
        return _exact_nonlinear(D, case["degree"], ca[0], ca[1], D["nodes"], values)
    P, b, on = _exact_elasticity(D, ca[0], ca[1], D["nodes"], values)
    return {"A": P.values(on), "b": b}
