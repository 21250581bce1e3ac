"""GPU parity at the sizes where a kernel's split into workgroups changes:
partly filled, exactly filled and single workgroups, one-cell problems and
constrained sets that leave some components free.  Against the oracle, to the
relative 1e-12 that the FP64 paths are held to everywhere (the sums here have
at most a few hundred terms of one sign pattern, 1e-14 at worst)."""
import numpy as np
import pytest

from oracle import cpu
from mifem import forms, problems
from mifem.fem import DirichletBC, Function, functionspace
from mifem.mesh import create_unit_cube

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _rel(x, ref):
    return np.linalg.norm(x - ref) / max(np.linalg.norm(ref), 1e-300)


def _poisson(n, k):
    mesh = create_unit_cube(n, jitter=0.2, seed=n)
    V = functionspace(mesh, ("P", k))
    kappa, f = Function(functionspace(mesh, ("DG", 0))), Function(V)
    rng = np.random.default_rng(k)
    kappa.x[:] = rng.uniform(1, 2, mesh.num_cells)
    f.x[:] = rng.uniform(-1, 1, V.size)
    return V, forms.stiffness(V, kappa), forms.source(V, f)


def _elasticity(n):
    P = problems.elasticity_p2(n)
    return P.V, P.a, P.L


def _some_dofs(V, share, seed):
    """A Dirichlet set of single scalar dofs: components of a node may stay free."""
    rng = np.random.default_rng(seed)
    dofs = np.flatnonzero(rng.random(V.size) < share).astype(np.int32)
    if dofs.size == 0:
        dofs = np.array([V.size // 2], dtype=np.int32)
    g = np.zeros(V.size)
    g[dofs] = rng.uniform(-1, 1, dofs.size)
    return DirichletBC(V, dofs, g)


@pytest.mark.parametrize("form,n,share", [
    ((1,), 1, 0.2), ((1,), 4, 0.02), ((2,), 3, 0.5), ((3,), 1, 0.0), ((3,), 4, 0.1),
    ((), 1, 0.1), ((), 3, 0.0), ((), 4, 0.3)])
def test_lifting_over_any_constrained_set(form, n, share):
    import cudolfinx as cufem
    print(f"[gpu-test] lifting {'P%d' % form if form else 'vector P2'} n={n} share={share}", flush=True)
    V, a, L = _poisson(n, *form) if form else _elasticity(n)
    bc = _some_dofs(V, share, 3)
    x0 = np.random.default_rng(9).uniform(-1, 1, V.size)
    af, Lf = cufem.form(a), cufem.form(L)
    asm = cufem.CUDAAssembler()
    b = asm.assemble_vector(Lf)
    xv = asm.create_vector(Lf)
    xv.data.upload(x0)
    asm.apply_lifting(b, [af], [asm.pack_bcs([bc])], x0=[xv], scale=-0.7)
    asm.synchronize()
    ref = cpu.OracleAssembler(L).assemble_vector()
    cpu.OracleAssembler(a).apply_lifting(ref, [bc], x0=x0, scale=-0.7)
    assert _rel(b.to_host(), ref) <= TOL


@pytest.mark.parametrize("degree,n,share,noalloc", [
    (1, 1, 0.3, False), (1, 5, 0.1, False), (2, 3, 0.05, True), (3, 1, 0.0, False), (3, 3, 0.2, True),
    (3, 4, 0.02, False)])
def test_hexahedral_lifting(degree, n, share, noalloc):
    """The sum-factorised lifting of Q1 to Q3 Helmholtz forms on jittered hexahedra."""
    import ctypes as C
    import cudolfinx as cufem
    from cudolfinx import _lib
    print(f"[gpu-test] hexahedral lifting Q{degree} n={n} share={share} noalloc={noalloc}", flush=True)
    P = problems.helmholtz_q3(n, seed=4, degree=degree)
    bc = _some_dofs(P.V, share, 5)
    x0 = np.random.default_rng(2).uniform(-1, 1, P.V.size)
    af, Lf = cufem.form(P.a), cufem.form(P.L)
    asm = cufem.CUDAAssembler()
    b, xv = asm.create_vector(Lf), asm.create_vector(Lf)
    xv.data.upload(x0)
    dbc = asm.pack_bcs([bc])
    if noalloc:
        _lib.check(_lib.lib().mf_apply_lifting_noalloc(
            (C.c_void_p * 1)(af.handle.value), 1, b.ptr, b.size,
            (C.c_void_p * 1)(dbc._get_cpp_bcs(P.V).handle.value), (C.c_void_p * 1)(xv.ptr.value), 0.9, None))
    else:
        asm.apply_lifting(b, [af], [dbc], x0=[xv], scale=0.9)
    asm.synchronize()
    ref = np.zeros(P.V.size)
    cpu.OracleAssembler(P.a).apply_lifting(ref, [bc], x0=x0, scale=0.9)
    assert _rel(b.to_host(), ref) <= TOL


@pytest.mark.parametrize("kernel", [0, 4])
@pytest.mark.parametrize("n,k", [(1, 1), (9, 1), (17, 1), (2, 3), (9, 2), (13, 3)])
def test_right_hand_side_rows_per_workgroup(n, k, kernel):
    import cudolfinx as cufem
    print(f"[gpu-test] right-hand side P{k} n={n} vector_kernel={kernel}", flush=True)
    V, _, L = _poisson(n, k)
    asm = cufem.CUDAAssembler()
    f = cufem.form(L, options={"vector_kernel": kernel})
    b = asm.assemble_vector(f)
    asm.synchronize()
    ref = cpu.OracleAssembler(L).assemble_vector()
    assert _rel(b.to_host(), ref) <= TOL
    asm.assemble_vector(f, b, zero=False)
    asm.synchronize()
    assert _rel(b.to_host(), 2 * ref) <= TOL


@pytest.mark.parametrize("which,n", [("elasticity", 1), ("elasticity", 4), ("hex", 1), ("hex", 5),
                                     ("shuffled", 4)])
def test_right_hand_side_in_blocks_of_cells(which, n):
    """Several components with a facet integral, 64 nodes per cell, and an order
    of the cells in which a block's cells share no rows."""
    import cudolfinx as cufem
    print(f"[gpu-test] right-hand side in blocks: {which} n={n}", flush=True)
    if which == "elasticity":
        L = _elasticity(n)[2]
    elif which == "hex":
        L = problems.helmholtz_q3(n, seed=2).L
    else:
        L = _poisson(n, 2)[2]
        L.integrals[0].entities = np.random.default_rng(0).permutation(L.integrals[0].entities)
    asm = cufem.CUDAAssembler()
    b = asm.assemble_vector(cufem.form(L, options={"vector_kernel": 4}))
    asm.synchronize()
    assert _rel(b.to_host(), cpu.OracleAssembler(L).assemble_vector()) <= TOL


@pytest.mark.parametrize("n,k,share", [(1, 1, 0.0), (3, 1, 0.2), (5, 1, 0.1), (1, 2, 0.3), (3, 2, 0.1)])
def test_gathered_element_tensors(n, k, share):
    """Forms without an owner kernel: element tensors summed by entry, with a
    Dirichlet set, against the per-entity kernel and the oracle; overwriting,
    then adding, then overwriting again; and bit-identical on repeat."""
    import cudolfinx as cufem
    from mifem.nonlinear import reference_test_forms
    print(f"[gpu-test] gathered tensors P{k} n={n} share={share}", flush=True)
    R = reference_test_forms(create_unit_cube(n, jitter=0.2, seed=1), k)
    a = R["matrix"][0]
    V = a.function_spaces[0]
    R["u"].x[:] = np.random.default_rng(4).uniform(-1, 1, V.size)
    bc = _some_dofs(V, share, 6)
    asm = cufem.CUDAAssembler()
    f = cufem.form(a)
    A = asm.assemble_matrix(f, bcs=[bc], diagonal=2.0)
    asm.synchronize()
    rp, cols, v = A.csr()
    o = cpu.OracleAssembler(a)
    orp, ocols, _, _ = o.sparsity()
    ref = o.assemble_matrix(orp, ocols, [bc], diagonal=2.0)
    assert np.array_equal(rp, orp) and np.array_equal(cols, ocols) and _rel(v, ref) <= TOL
    g = cufem.form(a, options={"matrix_kernel": 1})
    B = asm.assemble_matrix(g, bcs=[bc], diagonal=2.0)
    asm.synchronize()
    assert _rel(v, B.csr()[2]) <= TOL
    asm.assemble_matrix(f, A, bcs=[], zero=False)
    asm.synchronize()
    free = o.assemble_matrix(orp, ocols, [])
    assert _rel(A.csr()[2], ref + free) <= TOL
    asm.assemble_matrix(f, A, bcs=[bc], diagonal=2.0)
    asm.synchronize()
    assert np.array_equal(A.csr()[2], v)


def test_gathered_blocks_of_a_vector_form():
    """bs > 1 and different row and column Dirichlet sets (no owner kernel)."""
    import cudolfinx as cufem
    from cudolfinx import _lib
    V, a, _ = _elasticity(3)
    f = cufem.form(a)
    src = f.source()
    asm = cufem.CUDAAssembler()
    A = asm.create_matrix(f)
    b0, b1 = _some_dofs(V, 0.1, 1), _some_dofs(V, 0.2, 2)
    p0, p1 = asm.pack_bcs([b0]), asm.pack_bcs([b1])
    f.to_device()
    asm.pack_coefficients(f)
    _lib.check(_lib.lib().mf_assemble_matrix(f.handle, A.handle, p0._get_cpp_bcs(V).handle,
                                             p1._get_cpp_bcs(V).handle, 1.0, 1, None))
    asm.synchronize()
    assert "mf_mat_cell_0" in src
    o = cpu.OracleAssembler(a)
    rp, cols, _, _ = o.sparsity()
    full = o.assemble_matrix(rp, cols, [])
    rows = np.repeat(np.arange(V.size), np.diff(rp))
    m0, m1 = np.zeros(V.size, bool), np.zeros(V.size, bool)
    m0[b0.dofs], m1[b1.dofs] = True, True
    ref = np.where(m0[rows] | m1[cols], 0.0, full)
    ref[(rows == cols) & m0[rows]] = 1.0
    assert _rel(A.csr()[2], ref) <= TOL


@pytest.mark.parametrize("which,n", [("elasticity", 1), ("elasticity", 4), ("p1", 1), ("p1", 9), ("p3", 3),
                                     ("q3", 2), ("dg1", 2), ("two", 1), ("two", 5)])
def test_product_rows_of_any_length(which, n):
    """y = A x from the blocked pattern (three components) and row by row."""
    import scipy.sparse as sp
    import torch
    import cudolfinx as cufem
    print(f"[gpu-test] product {which} n={n}", flush=True)
    if which == "elasticity":
        a = _elasticity(n)[1]
    elif which == "q3":
        a = problems.helmholtz_q3(n).a
    elif which == "dg1":
        a = problems.dg_plaplace(n).a
    elif which == "two":
        V = functionspace(create_unit_cube(n), ("P", 1), shape=(2,))
        name = "tabulate_tensor_integral_two"
        body = "{\n  for (int i = 0; i < 8; ++i)\n    for (int j = 0; j < 8; ++j) A[8 * i + j] += 1.0 / (1 + i + 2 * j);\n}\n"
        a = forms.Form(2, [V, V], [forms.Integral("cell", -1, np.arange(V.mesh.num_cells, dtype=np.int32),
                                                  name, forms._SIG.format(name=name) + "\n" + body)])
    else:
        a = _poisson(n, int(which[1]))[1]
    asm = cufem.CUDAAssembler()
    A = asm.assemble_matrix(cufem.form(a))
    asm.synchronize()
    rp, cols, vals = A.csr()
    x = np.random.default_rng(1).uniform(-1, 1, A.ncols)
    y = torch.full((A.nrows,), 7.0, dtype=torch.float64, device="cuda")
    A.mult(torch.from_numpy(x).cuda(), y)
    S = sp.csr_matrix((vals, cols, rp), shape=(A.nrows, A.ncols))
    # at most 400 products per row, each rounded once: 400 eps of the absolute sums
    assert np.all(np.abs(y.cpu().numpy() - S @ x) <= 400 * 2.2e-16 * (abs(S) @ np.abs(x)) + 1e-300)


@pytest.mark.parametrize("part", [(0, 1), (0, 0.5), (0.5, 0.625), (0.99, 1)])
@pytest.mark.parametrize("degree,n", [(1, 11), (1, 12), (1, 21), (2, 9), (2, 12)])
def test_product_with_rows_empty(degree, n, part):
    """y = A x with the entries in one part of the rows: every row is written once,
    in each order of the workgroups and for every width."""
    import dataclasses
    import scipy.sparse as sp
    import torch
    import cudolfinx as cufem
    print(f"[gpu-test] product over a part: P{degree} n={n} {part}", flush=True)
    V, a, L = _poisson(n, degree)
    cells = np.arange(*(int(p * 6 * n**3) for p in part), dtype=np.int32)
    a = dataclasses.replace(a, integrals=[dataclasses.replace(a.integrals[0], entities=cells)])
    asm = cufem.CUDAAssembler()
    A = asm.assemble_matrix(cufem.form(a))
    asm.synchronize()
    rp, cols, vals = A.csr()
    x = np.random.default_rng(1).uniform(-1, 1, A.ncols)
    y = torch.full((A.nrows,), 7.0, dtype=torch.float64, device="cuda")
    A.mult(torch.from_numpy(x).cuda(), y)
    S = sp.csr_matrix((vals, cols, rp), shape=(A.nrows, A.ncols))
    # at most 400 products per row, each rounded once: 400 eps of the absolute sums
    assert np.all(np.abs(y.cpu().numpy() - S @ x) <= 400 * 2.2e-16 * (abs(S) @ np.abs(x)) + 1e-300)


@pytest.mark.parametrize("prec,tol", [(64, TOL), (32, 1e-6)])
@pytest.mark.parametrize("n,share,subset", [(1, 0.1, False), (2, 0.0, False), (3, 0.3, True), (5, 0.05, True),
                                            (7, 0.1, False)])
def test_hexahedral_owner_chunks(n, share, subset, prec, tol):
    """Q3 matrices from one cell to more chunks than resident workgroups per XCD,
    with Dirichlet rows, over all cells or a subdomain (rows and chunks without
    cells), overwriting and adding."""
    import dataclasses
    import cudolfinx as cufem
    print(f"[gpu-test] Q3 owner chunks n={n} share={share} subset={subset} precision={prec}", flush=True)
    P = problems.helmholtz_q3(n, seed=8)
    a = P.a
    if subset:
        I = a.integrals[0]
        keep = np.sort(np.random.default_rng(n).choice(n ** 3, size=n ** 3 // 3, replace=False)).astype(np.int32)
        a = dataclasses.replace(a, integrals=[dataclasses.replace(I, entities=keep)])
    bc = _some_dofs(P.V, share, 3)
    asm = cufem.CUDAAssembler()
    f = cufem.form(a, options={"matrix_kernel": 2, "precision": prec})
    A = asm.assemble_matrix(f, bcs=[bc], diagonal=1.5)
    asm.synchronize()
    rp, cols, v = A.csr()
    o = cpu.OracleAssembler(a)
    orp, ocols, _, _ = o.sparsity()
    ref = o.assemble_matrix(orp, ocols, [bc], diagonal=1.5)
    assert np.array_equal(rp, orp) and np.array_equal(cols, ocols)
    # FP32 element arithmetic keeps its 1e-6; the diagonal entries are exact
    scale = np.linalg.norm(o.assemble_matrix(orp, ocols, []))
    assert np.linalg.norm(v - ref) <= tol * max(scale, np.linalg.norm(ref))
    asm.assemble_matrix(f, A, bcs=[bc], diagonal=1.5, zero=False)
    asm.synchronize()
    ref = o.assemble_matrix(orp, ocols, [bc], diagonal=1.5, values=ref.copy())
    assert np.linalg.norm(A.csr()[2] - ref) <= 2 * tol * max(scale, np.linalg.norm(ref))


@pytest.mark.parametrize("which", ["hex", "hex32", "pipe", "owner", "dg0"])
def test_values_beside_rows_without_entries(which):
    """Chunks without values that start on an odd entry, between and behind others:
    they write nothing."""
    import dataclasses
    import cudolfinx as cufem
    print(f"[gpu-test] values beside empty rows: {which}", flush=True)
    if which.startswith("hex"):
        P = problems.helmholtz_q3(8, seed=8)
        V, a = P.V, P.a
        mid = V.mesh.x[V.mesh.cells].mean(axis=1)
        low = np.flatnonzero((mid < 0.25).all(axis=1))           # 2 x 2 x 2 cells: one row of 343
        cells = np.concatenate([low, np.flatnonzero((mid > 0.7).all(axis=1))[:1]])
    elif which == "dg0":
        V = functionspace(create_unit_cube(7), ("DG", 0))
        a = forms.mass(V)
        cells = np.array([3, 70, 71, 900, 901, 902, 903, 904, 1500], dtype=np.int32)
    else:
        V, a = _poisson(9, 1)[:2]
        cells = np.r_[0:2, 6:9, 3000:3002, 3900:3902]
    cells = np.sort(cells).astype(np.int32)
    a = dataclasses.replace(a, integrals=[dataclasses.replace(a.integrals[0], entities=cells)])
    o = cpu.OracleAssembler(a)
    orp, ocols, _, _ = o.sparsity()
    empty = np.diff(orp) == 0
    runs = np.split(np.arange(empty.size), np.flatnonzero(np.diff(empty.astype(int))) + 1)
    odd = [r for r in runs if empty[r[0]] and r.size >= 128 and orp[r[0]] % 2]
    assert odd, which
    options = {"hex": {"matrix_kernel": 2}, "hex32": {"matrix_kernel": 2, "precision": 32},
               "pipe": {"matrix_kernel": 2, "owner_pipe": 1}, "owner": {"matrix_kernel": 2}, "dg0": {}}[which]
    f = cufem.form(a, options=options)
    asm = cufem.CUDAAssembler()
    ref = o.assemble_matrix(orp, ocols, [])
    A = asm.assemble_matrix(f)
    for _ in range(3):
        asm.assemble_matrix(f, A)
        asm.synchronize()
        rp, cols, v = A.csr()
        assert np.array_equal(rp, orp) and np.array_equal(cols, ocols)
        assert np.abs(v - ref).max() <= (1e-6 if which == "hex32" else TOL) * np.abs(ref).max()


@pytest.mark.parametrize("k,m,n,subset", [(1, 2, 1, False), (1, 3, 9, True), (2, 2, 3, False), (3, 4, 1, False),
                                          (3, 4, 5, True), (3, 4, 13, False), (4, 6, 3, False), (5, 5, 2, True),
                                          (6, 7, 1, False)])
def test_hexahedral_source(k, m, n, subset):
    """Q_k sources on hexahedra against the per-entity kernel, and the oracle where it
    takes the degree: more and fewer points than nodes per direction, a partial last
    block, a subdomain, a degree past the kernel's, a sum of two sources, and its
    second one alone, whose constant is not the form's first."""
    import dataclasses
    import cudolfinx as cufem
    from mifem import forms
    from mifem.fem import Constant, functionspace
    from mifem.mesh import create_unit_cube
    print(f"[gpu-test] Q{k} source m={m} n={n} subset={subset}", flush=True)
    V = functionspace(create_unit_cube(n, "hexahedron", jitter=0.2, seed=3), ("P", k))
    L = forms.hex_source(V, Constant(1.7), qpoints_per_dir=m)
    M = forms.hex_source(V, Constant(-0.3), qpoints_per_dir=m - 1)
    if subset:
        keep = np.sort(np.random.default_rng(n).choice(n ** 3, size=n ** 3 // 2, replace=False)).astype(np.int32)
        L = dataclasses.replace(L, integrals=[dataclasses.replace(L.integrals[0], entities=keep)])
    S = forms.linear_sum(M, L)
    asm = cufem.CUDAAssembler()
    for F in (L, S, dataclasses.replace(S, integrals=S.integrals[1:])):
        f = cufem.form(F)
        b = asm.assemble_vector(f)
        asm.synchronize()
        per_entity = asm.assemble_vector(cufem.form(F, options={"vector_kernel": 1}))
        asm.synchronize()
        ref = per_entity.to_host()
        assert _rel(b.to_host(), ref) <= TOL
        if k <= 3 and m <= 4:
            assert _rel(b.to_host(), cpu.OracleAssembler(F).assemble_vector()) <= TOL
        asm.assemble_vector(f, b, zero=False)
        asm.synchronize()
        assert _rel(b.to_host(), 2 * ref) <= TOL


@pytest.mark.parametrize("n", [1, 2, 3, 5])
def test_fused_system_adds_with_dirichlet_rows(n):
    """J, F and E of DG1 in blocks of 64 cells (partial, exact and several, segments
    that start at odd values' alignment): overwriting, then adding, with Dirichlet rows."""
    import torch
    import cudolfinx as cufem
    from mifem.dgforms import sipg_energy
    print(f"[gpu-test] DG1 system n={n}", flush=True)
    P = problems.dg_plaplace(n)
    P.extras["u"].x[:] = np.random.default_rng(n).uniform(-1, 1, P.V.size)
    bc = _some_dofs(P.V, 0.2, 5)
    J, F, E_ = cufem.form(P.a), cufem.form(P.L), cufem.form(sipg_energy(P.V, P.extras["u"]))
    asm = cufem.CUDAAssembler()
    A, b = asm.create_matrix(J), asm.create_vector(F)
    system, ev = cufem.CUDASystem(J, F, E_), torch.zeros(1, dtype=torch.float64, device="cuda")
    o = cpu.OracleAssembler(P.a)
    rp, cols, _, _ = o.sparsity()
    ref, rhs = o.assemble_matrix(rp, cols, [bc], diagonal=2.5), cpu.OracleAssembler(P.L).assemble_vector()
    for times in (1, 2):
        system.assemble(asm, A, b, ev, bcs=asm.pack_bcs([bc]), diagonal=2.5, zero=times == 1)
        asm.synchronize()
        assert _rel(A.csr()[2], ref) <= TOL
        assert _rel(b.to_host(), times * rhs) <= TOL
        ref = o.assemble_matrix(rp, cols, [bc], diagonal=2.5, values=ref.copy())


@pytest.mark.parametrize("which,times", [("vector", 1), ("vector", 5), ("vector", 6), ("vector", 8), ("vector", 17),
                                         (2, 10), (2, 12), (3, 11), (3, 17)])
def test_matrix_rows_with_many_cells(which, times):
    """Rows around the numbers of (cell, row) pairs at which the owner kernel's shape
    changes (128 vector, 256 scalar) and past its largest (384): every cell of a cube
    listed several times, so that its inner node has 24 cells as often."""
    import dataclasses
    import cudolfinx as cufem
    print(f"[gpu-test] matrix {which} with cells listed {times} times", flush=True)
    V, a, _ = _elasticity(2) if which == "vector" else _poisson(2, which)
    ents = np.repeat(np.arange(V.mesh.num_cells, dtype=np.int32), times)
    a = dataclasses.replace(a, integrals=[dataclasses.replace(a.integrals[0], entities=ents)])
    bc = _some_dofs(V, 0.1, 3)
    asm = cufem.CUDAAssembler()
    A = asm.assemble_matrix(cufem.form(a), bcs=[bc])
    asm.synchronize()
    o = cpu.OracleAssembler(a)
    rp, cols, _, _ = o.sparsity()
    ref = o.assemble_matrix(rp, cols, [bc])
    assert _rel(A.csr()[2], ref) <= TOL


@pytest.mark.parametrize("n,count", [(1, 1), (3, 2), (2, 3), (4, 4), (3, 5), (2, 8), (3, 9), (2, 17)])
def test_packed_coefficients_of_one_form(n, count):
    """Coefficients of widths 1, 4, 10 and 12 packed together, more of them than one
    launch takes; then some of them changed: b_i = (i + 1) sum_k (k + 1) w_k."""
    import cudolfinx as cufem
    from mifem.forms import _SIG, CELL, Form, Integral
    print(f"[gpu-test] {count} coefficients on n={n}", flush=True)
    mesh = create_unit_cube(n, jitter=0.1, seed=2)
    V = functionspace(mesh, ("P", 1))
    spaces = [functionspace(mesh, ("DG", 0)), V, functionspace(mesh, ("P", 2)), functionspace(mesh, ("P", 1), (3,))]
    w = [Function(spaces[k % 4]) for k in range(count)]
    rng = np.random.default_rng(count)
    for f in w:
        f.x[:] = rng.uniform(-1, 1, f.x.size)
    width = sum(f.function_space.element.ndofs * f.function_space.bs for f in w)
    name = f"tabulate_tensor_integral_packs_{count}"
    src = _SIG.format(name=name) + f"""
{{
  double s = 0.0;
  for (int k = 0; k < {width}; ++k) s += (k + 1) * w[k];
  for (int i = 0; i < 4; ++i) A[i] += (i + 1) * s;
}}
"""
    cells = np.arange(mesh.num_cells, dtype=np.int32)
    L = Form(1, [V], [Integral(CELL, -1, cells, name, src, None, {})], w, [], "packs")

    def reference():
        packed = []
        for f in w:
            S = f.function_space
            dofs = S.bs * np.repeat(S.dofmap, S.bs, axis=1) + np.tile(np.arange(S.bs), S.element.ndofs)
            packed.append(f.x[dofs])
        s = np.concatenate(packed, axis=1) @ np.arange(1.0, width + 1)
        b = np.zeros(V.size)
        np.add.at(b, V.dofmap, s[:, None] * np.arange(1.0, 5.0))
        return b

    asm = cufem.CUDAAssembler()
    form = cufem.form(L)
    b = asm.assemble_vector(form)
    asm.synchronize()
    assert _rel(b.to_host(), reference()) <= TOL
    for f in w[::2]:
        f.x[:] = rng.uniform(-1, 1, f.x.size)
    form.to_device()
    b = asm.assemble_vector(form, b)
    asm.synchronize()
    assert _rel(b.to_host(), reference()) <= TOL


@pytest.mark.parametrize("prec,tol", [(64, TOL), (32, 1e-6), (16, 2e-2)])
def test_hexahedral_accumulator_of_odd_length(prec, tol):
    """chunk_values = 343, which the row of an inner vertex (7^3 columns) fills to
    the last value, after a kernel that leaves sums in LDS."""
    import cudolfinx as cufem
    print(f"[gpu-test] Q3 owner chunks of 343 values, precision={prec}", flush=True)
    P = problems.helmholtz_q3(4, seed=8)
    asm = cufem.CUDAAssembler()
    f = cufem.form(P.a, options={"matrix_kernel": 2, "precision": prec, "chunk_values": 343})
    A = asm.create_matrix(f)
    o = cpu.OracleAssembler(P.a)
    rp, cols, _, _ = o.sparsity()
    ref = o.assemble_matrix(rp, cols, [])
    assert np.diff(rp).max() == 343
    fill = cufem.form(_elasticity(9)[2], options={"vector_kernel": 4})
    for _ in range(4):
        asm.assemble_vector(fill)
        asm.assemble_matrix(f, A)
        asm.synchronize()
        assert _rel(A.csr()[2], ref) <= tol


@pytest.mark.parametrize("options", [{"hex_block": 64}, {"chunk_rows": 256}, {"chunk_rows": 1500, "chunk_values": 6000},
                                     {"hex_block": 64, "owner_nb": 70, "owner_lds": 160000}])
@pytest.mark.parametrize("prec,tol", [(64, TOL), (32, 1e-6)])
def test_hexahedral_chunks_of_more_rows_than_threads(options, prec, tol):
    """Workgroups of fewer threads than a chunk has rows or a batch has cells,
    over a subdomain (rows without cells fill chunks with hundreds of rows)."""
    import dataclasses
    import cudolfinx as cufem
    print(f"[gpu-test] Q3 owner chunks {options} precision={prec}", flush=True)
    P = problems.helmholtz_q3(5, seed=8)
    I = P.a.integrals[0]
    a = dataclasses.replace(P.a, integrals=[dataclasses.replace(I, entities=np.arange(0, 125, 3, dtype=np.int32))])
    bc = _some_dofs(P.V, 0.1, 3)
    asm = cufem.CUDAAssembler()
    f = cufem.form(a, options={"matrix_kernel": 2, "precision": prec, **options})
    A = asm.assemble_matrix(f, bcs=[bc], diagonal=1.5)
    asm.synchronize()
    o = cpu.OracleAssembler(a)
    rp, cols, _, _ = o.sparsity()
    ref = o.assemble_matrix(rp, cols, [bc], diagonal=1.5)
    scale = np.linalg.norm(o.assemble_matrix(rp, cols, []))
    assert np.linalg.norm(A.csr()[2] - ref) <= tol * max(scale, np.linalg.norm(ref))


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("form", [(1,), (2,), (3,), ()])
def test_lifting_of_zero_values_keeps_nan(form, noalloc):
    """A constrained value of zero lifts the NaN of a cell's tensor, as any other
    value does (only one constrained dof, in another cell, is not zero)."""
    import ctypes as C
    import cudolfinx as cufem
    from cudolfinx import _lib
    print(f"[gpu-test] NaN coefficient under lifting: {'P%d' % form if form else 'vector P2'} "
          f"noalloc={noalloc}", flush=True)
    V, a, L = _poisson(4, *form) if form else _elasticity(4)
    a.coefficients[0].x[7] = np.nan
    cells = V.dofmap
    bs = V.bs
    dofs = np.unique(np.concatenate([bs * cells[7][:2], bs * cells[-1][-2:]])).astype(np.int32)
    far = int(bs * cells[-1][-1])
    assert far // bs not in cells[7]
    g = np.zeros(V.size)
    g[far] = 1.0
    bc = DirichletBC(V, dofs, g)
    af, Lf = cufem.form(a), cufem.form(L)
    asm = cufem.CUDAAssembler()
    dbc = asm.pack_bcs([bc])
    b = asm.create_vector(Lf)
    asm.pack_coefficients(af)
    if noalloc:
        _lib.check(_lib.lib().mf_apply_lifting_noalloc(
            (C.c_void_p * 1)(af.handle.value), 1, b.ptr, b.size,
            (C.c_void_p * 1)(dbc._get_cpp_bcs(V).handle.value), None, 1.0, None))
    else:
        asm.apply_lifting(b, [af], [dbc])
    asm.synchronize()
    got, ref = b.to_host(), np.zeros(V.size)
    cpu.OracleAssembler(a).apply_lifting(ref, [bc])
    nan = np.isnan(ref)
    assert nan.any() and not nan.all()
    assert np.array_equal(np.isnan(got), nan)
    assert _rel(got[~nan], ref[~nan]) <= TOL


@pytest.mark.parametrize("form,n,share", [
    ((1,), 1, 0.2), ((1,), 5, 0.02), ((1,), 5, 1.0), ((2,), 3, 0.5), ((3,), 1, 0.0), ((3,), 4, 0.1), ((), 3, 0.3)])
def test_lifting_without_a_list_on_the_host(form, n, share):
    """mf_apply_lifting_noalloc: workgroups past the list's end, the last one
    partly filled, every cell listed."""
    import ctypes as C
    import cudolfinx as cufem
    from cudolfinx import _lib
    print(f"[gpu-test] noalloc lifting {'P%d' % form if form else 'vector P2'} n={n} share={share}", flush=True)
    V, a, L = _poisson(n, *form) if form else _elasticity(n)
    bc = _some_dofs(V, share, 3)
    x0 = np.random.default_rng(9).uniform(-1, 1, V.size)
    af, Lf = cufem.form(a), cufem.form(L)
    asm = cufem.CUDAAssembler()
    dbc = asm.pack_bcs([bc])
    b, xv = asm.create_vector(Lf), asm.create_vector(Lf)
    xv.data.upload(x0)
    asm.pack_coefficients(af)
    _lib.check(_lib.lib().mf_apply_lifting_noalloc(
        (C.c_void_p * 1)(af.handle.value), 1, b.ptr, b.size,
        (C.c_void_p * 1)(dbc._get_cpp_bcs(V).handle.value), (C.c_void_p * 1)(xv.ptr.value), -0.7, None))
    asm.synchronize()
    ref = np.zeros(V.size)
    cpu.OracleAssembler(a).apply_lifting(ref, [bc], x0=x0, scale=-0.7)
    assert _rel(b.to_host(), ref) <= TOL


@pytest.mark.parametrize("sets", ["rows", "columns", "both"])
@pytest.mark.parametrize("which,n", [("tet", 1), ("tet", 4), ("triangle", 1), ("triangle", 9)])
def test_fused_system_masks_rows_and_columns(which, n, sets):
    """Row and column sets of their own (four and three dofs per cell): the masks of
    a cell's neighbours, overwriting and adding."""
    import cudolfinx as cufem
    from cudolfinx import _lib
    from mifem.mesh import create_unit_square
    from mifem.nonlinear import reference_test_forms
    print(f"[gpu-test] DG1 system on {which} n={n}, {sets}", flush=True)
    if which == "tet":
        P = problems.dg_plaplace(n)
        a, L, u = P.a, P.L, P.extras["u"]
    else:
        R = reference_test_forms(create_unit_square(n, n), 1)
        a, L, u = R["matrix"][2], R["vector"][2], R["u_dg"]
    V = a.function_spaces[0]
    u.x[:] = np.random.default_rng(n).uniform(-1, 1, V.size)
    b0, b1 = _some_dofs(V, 0.1, 1), _some_dofs(V, 0.05, 2)
    J, F = cufem.form(a), cufem.form(L)
    asm = cufem.CUDAAssembler()
    p0, p1 = asm.pack_bcs([b0] if sets != "columns" else []), asm.pack_bcs([b1] if sets != "rows" else [])
    A, b, S = asm.create_matrix(J), asm.create_vector(F), cufem.CUDASystem(J, F)
    asm.pack_coefficients(J)
    o = cpu.OracleAssembler(a)
    rp, cols, _, _ = o.sparsity()
    full, rhs = o.assemble_matrix(rp, cols, []), cpu.OracleAssembler(L).assemble_vector()
    rows = np.repeat(np.arange(V.size), np.diff(rp))
    m0, m1 = np.zeros(V.size, bool), np.zeros(V.size, bool)
    m0[b0.dofs], m1[b1.dofs] = sets != "columns", sets != "rows"
    for times in (1, 2):
        _lib.check(_lib.lib().mf_system_assemble(S.handle, A.handle, p0._get_cpp_bcs(V).handle,
                                                 p1._get_cpp_bcs(V).handle, 2.5, b.ptr, b.size, None,
                                                 int(times == 1), None))
        asm.synchronize()
        ref = np.where(m0[rows] | m1[cols], 0.0, times * full)
        ref[(rows == cols) & m0[rows]] = 2.5
        assert _rel(A.csr()[2], ref) <= TOL
        assert _rel(b.to_host(), times * rhs) <= TOL


@pytest.mark.parametrize("degree,bs,n,times", [(1, 3, 1, 1), (1, 3, 5, 1), (1, 3, 11, 1), (1, 3, 2, 8), (1, 3, 2, 12),
                                               (1, 1, 4, 1), (1, 1, 12, 1), (2, 1, 3, 1), (2, 1, 8, 1), (2, 1, 2, 12),
                                               (3, 1, 2, 1)])
def test_default_shapes_of_sums_over_points(degree, bs, n, times):
    """The owner kernel of forms without a reference tensor, by degree and components:
    meshes on both sides of the size at which a chunk's pairs change, and cells listed
    several times (rows of more than 128 and 256 cells); the owner kernel runs
    (matrix_kernel = 2 refuses any other)."""
    import dataclasses
    import cudolfinx as cufem
    print(f"[gpu-test] default shape P{degree} x {bs} n={n} cells listed {times} times", flush=True)
    if bs == 3:
        mesh = create_unit_cube(n, jitter=0.2, seed=n)
        V, D = functionspace(mesh, ("P", degree), shape=(3,)), functionspace(mesh, ("DG", 0))
        mu, lam = Function(D), Function(D)
        mu.x[:], lam.x[:] = np.random.default_rng(n).uniform(1, 2, (2, mesh.num_cells))
        a = forms.elasticity(V, mu, lam)
    else:
        V, a, _ = _poisson(n, degree)
        I = a.integrals[0]
        a = dataclasses.replace(a, integrals=[dataclasses.replace(
            I, staged=dataclasses.replace(I.staged, trace_only=False))])
    ents = np.repeat(np.arange(V.mesh.num_cells, dtype=np.int32), times)
    a = dataclasses.replace(a, integrals=[dataclasses.replace(a.integrals[0], entities=ents)])
    bc = _some_dofs(V, 0.1, 3)
    asm = cufem.CUDAAssembler()
    A = asm.assemble_matrix(cufem.form(a, options={"matrix_kernel": 2}), bcs=[bc], diagonal=2.0)
    asm.synchronize()
    o = cpu.OracleAssembler(a)
    rp, cols, _, _ = o.sparsity()
    assert _rel(A.csr()[2], o.assemble_matrix(rp, cols, [bc], diagonal=2.0)) <= TOL


def _replays(g, launches, state, eager, check):
    """Each replay of graph g with another state, between eager runs of the same
    calls, against them."""
    import torch
    for k in range(launches):
        state(k)
        torch.cuda.synchronize()
        g.launch()
        torch.cuda.synchronize()
        got = check()
        state(k)
        eager()
        torch.cuda.synchronize()
        ref = check()
        assert _rel(got, ref) <= TOL, k
        state(k + launches)
        eager()
        torch.cuda.synchronize()


@pytest.mark.parametrize("warm,captured", [(True, False), (False, True), (True, True)])
def test_capture_of_a_gathered_matrix_after_either_mode(warm, captured):
    """One uncaptured call, overwriting or adding, is enough for a captured one of
    either kind (forms without an owner kernel)."""
    import torch
    import cudolfinx as cufem
    from mifem.nonlinear import reference_test_forms
    print(f"[gpu-test] gathered matrix: eager zero={warm}, captured zero={captured}", flush=True)
    R = reference_test_forms(create_unit_cube(3, jitter=0.2, seed=1), 2)
    a = R["matrix"][0]
    V = a.function_spaces[0]
    s = torch.cuda.Stream()
    asm = cufem.CUDAAssembler(stream=s)
    f = cufem.form(a)
    u = torch.zeros(V.size, dtype=torch.float64, device="cuda")
    f.set_coefficient_device(0, u.data_ptr(), V.size)
    A = asm.create_matrix(f)
    asm.assemble_matrix(f, A, zero=warm)
    asm.synchronize()
    g = cufem.CUDAGraph(s)
    with g:
        asm.assemble_matrix(f, A, zero=captured)

    def state(k):
        u.copy_(torch.from_numpy(np.random.default_rng(k).uniform(-1, 1, V.size)))
        h = A.device_arrays()[2]
        from cudolfinx import _lib
        _lib.check(_lib.lib().mf_zero(asm._ctx.handle, h, A.nnz, asm._stream))

    _replays(g, 3, state, lambda: asm.assemble_matrix(f, A, zero=captured), lambda: A.csr()[2].copy())


@pytest.mark.parametrize("zero", [True, False])
def test_capture_of_a_right_hand_side_without_an_eager_call(zero):
    """Forms of more than 32 nodes per cell need no schedule, so their first call
    may be captured."""
    import torch
    import cudolfinx as cufem
    print(f"[gpu-test] Q3 source, first call captured, zero={zero}", flush=True)
    P = problems.helmholtz_q3(3, seed=2)
    s = torch.cuda.Stream()
    asm = cufem.CUDAAssembler(stream=s)
    f = cufem.form(P.L)
    b = asm.create_vector(f)
    asm.assemble_vector(cufem.form(P.L, options={"vector_kernel": 1}), b)   # b holds something
    asm.synchronize()
    g = cufem.CUDAGraph(s)
    with g:
        asm.assemble_vector(f, b, zero=zero)
    ref = cpu.OracleAssembler(P.L).assemble_vector()
    for k in range(1, 4):
        g.launch()
        asm.synchronize()
        assert _rel(b.to_host(), ref if zero else (2 * k) * ref) <= TOL
        asm.assemble_vector(f, b, zero=zero)                 # eager calls between the replays
        asm.synchronize()
        assert _rel(b.to_host(), ref if zero else (2 * k + 1) * ref) <= TOL


@pytest.mark.parametrize("warm,captured", [(64, 32), (32, 64), (16, 64), (64, 16)])
def test_capture_of_another_precision(warm, captured):
    """Q3 matrices: one uncaptured call in one precision is enough for a captured
    one in another (precision is set between calls)."""
    import torch
    import cudolfinx as cufem
    print(f"[gpu-test] Q3 eager FP{warm}, captured FP{captured}", flush=True)
    P = problems.helmholtz_q3(3, seed=2)
    s = torch.cuda.Stream()
    asm = cufem.CUDAAssembler(stream=s)
    f = cufem.form(P.a, options={"precision": warm})
    bcs = asm.pack_bcs([_some_dofs(P.V, 0.1, 3)])
    A = asm.create_matrix(f)
    asm.assemble_matrix(f, A, bcs=bcs)
    asm.synchronize()
    f.set_option("precision", captured)
    g = cufem.CUDAGraph(s)
    with g:
        asm.assemble_matrix(f, A, bcs=bcs)
    asm.assemble_matrix(f, A, bcs=bcs)                       # the schedule of its own
    asm.synchronize()
    ref = A.csr()[2].copy()
    o = cpu.OracleAssembler(P.a)
    rp, cols, _, _ = o.sparsity()
    tol = {64: TOL, 32: 1e-6, 16: 2e-2}[captured]
    assert _rel(ref, o.assemble_matrix(rp, cols, [_some_dofs(P.V, 0.1, 3)])) <= tol
    for _ in range(3):
        g.launch()
        asm.synchronize()
        # the same element arithmetic, summed in another order
        assert _rel(A.csr()[2], ref) <= TOL
        f.set_option("precision", warm)
        asm.assemble_matrix(f, A, bcs=bcs)
        asm.synchronize()
        f.set_option("precision", captured)


def test_forms_on_one_matrix_share_a_gather_workspace():
    """A program that builds its form again and again for a matrix it keeps: device
    memory grows by a form's own tables, not by another workspace."""
    import dataclasses
    import torch
    import cudolfinx as cufem
    print("[gpu-test] forms rebuilt against one matrix: device memory", flush=True)
    V, a, _ = _elasticity(8)
    a = dataclasses.replace(a, integrals=[dataclasses.replace(a.integrals[0], staged=None)])
    asm = cufem.CUDAAssembler()
    first = cufem.form(a)
    A = asm.assemble_matrix(first)
    asm.synchronize()
    ref = A.csr()[2].copy()
    workspace = 8 * 900 * V.mesh.num_cells                   # the element tensors
    before = torch.cuda.mem_get_info()[0]
    for _ in range(6):
        f = cufem.form(a)
        asm.assemble_matrix(f, A)
        asm.synchronize()
        assert _rel(A.csr()[2], ref) <= TOL
        del f
    used = before - torch.cuda.mem_get_info()[0]
    assert used < 3 * workspace, (used, workspace)
    asm.assemble_matrix(first, A)                            # its plan still holds what it needs
    asm.synchronize()
    assert _rel(A.csr()[2], ref) <= TOL


@pytest.mark.parametrize("n,share", [(3, 30), (3, 70), (5, 200), (7, 2058)])
def test_matrix_with_a_node_that_many_cells_share(n, share):
    """Entries of 30 to 2,058 contributions, on both sides of the line between the
    gather and the per-entity kernel."""
    import cudolfinx as cufem
    print(f"[gpu-test] P1 mass n={n}, one node in {share} cells", flush=True)
    V = functionspace(create_unit_cube(n, jitter=0.2, seed=1), ("P", 1))
    d = V.dofmap.copy()
    for c in np.random.default_rng(1).permutation(d.shape[0])[:share]:
        if 0 not in d[c]:
            d[c, 3] = 0
    V._dofmap = d
    a = forms.mass(V)
    bc = _some_dofs(V, 0.1, 3)
    asm = cufem.CUDAAssembler()
    f = cufem.form(a)
    A = asm.assemble_matrix(f, bcs=[bc], diagonal=2.0)
    asm.synchronize()
    o = cpu.OracleAssembler(a)
    rp, cols, _, _ = o.sparsity()
    ref = o.assemble_matrix(rp, cols, [bc], diagonal=2.0)
    assert _rel(A.csr()[2], ref) <= TOL
    asm.assemble_matrix(f, A, zero=False)
    asm.synchronize()
    assert _rel(A.csr()[2], ref + o.assemble_matrix(rp, cols, [])) <= TOL


def _two_components(n):
    """An unsymmetric form of two components per node that depends on the cell's
    coordinates, and its element tensors by numpy."""
    V = functionspace(create_unit_cube(n, jitter=0.2, seed=n), ("P", 1), shape=(2,))
    name = "tabulate_tensor_integral_unsymmetric2"
    body = ("{\n  for (int i = 0; i < 8; ++i)\n    for (int j = 0; j < 8; ++j)\n"
            "      A[8 * i + j] += (1 + i + 3 * j) * coordinate_dofs[0] + (2 + i * j) * coordinate_dofs[4] + 0.5 * i;\n}\n")
    a = forms.Form(2, [V, V], [forms.Integral("cell", -1, np.arange(V.mesh.num_cells, dtype=np.int32), name,
                                              forms._SIG.format(name=name) + "\n" + body)])
    i, j = np.meshgrid(np.arange(8), np.arange(8), indexing="ij")
    x = V.mesh.x[V.mesh.cells]
    T = ((1 + i + 3 * j) * x[:, 0, 0, None, None] + (2 + i * j) * x[:, 1, 1, None, None] + 0.5 * i)
    return V, V, a, T


def _at_pattern(V, W, rp, cols, T):
    """The CSR values of the sum of element tensors T (one per cell)."""
    D = np.zeros((V.size, W.size))
    for r, c, t in zip(V.unrolled_dofmap(), W.unrolled_dofmap(), T):
        D[np.ix_(r, c)] += t
    v = D[np.repeat(np.arange(V.size), np.diff(rp)), cols]
    assert np.count_nonzero(D) == np.count_nonzero(v)
    return v


@pytest.mark.parametrize("sets", ["none", "equal", "different"])
@pytest.mark.parametrize("which,n", [("three", 1), ("three", 3), ("two", 1), ("two", 4), ("rectangular", 3),
                                     ("facets", 1), ("facets", 3), ("interior", 2), ("triangle", 5)])
def test_gathered_blocks_spaces_and_facets(which, n, sets):
    """The gather (mf_ten_* is in the source and no owner kernel) of blocks of 3 x 3 and
    2 x 2, of different row and column spaces and of two-cell entities (facets of a
    continuous space, whose cells share rows), and a discontinuous space out of order
    (no gather), against the oracle (numpy for the 2 x 2 form): overwriting, then
    adding."""
    import dataclasses
    import cudolfinx as cufem
    from cudolfinx import _lib
    from mifem.mesh import create_unit_square
    from mifem.nonlinear import reference_test_forms
    print(f"[gpu-test] gathered {which} n={n}, {sets} Dirichlet sets", flush=True)
    T = None
    if which == "three":
        V, a, _ = _elasticity(n)
        W = V
        a = dataclasses.replace(a, integrals=[dataclasses.replace(a.integrals[0], staged=None)])
    elif which == "two":
        V, W, a, T = _two_components(n)
    elif which == "rectangular":
        m = create_unit_cube(n, jitter=0.2, seed=n)
        V, W = functionspace(m, ("P", 2)), functionspace(m, ("P", 1))
        a = forms.mass(V, W)
    elif which == "facets":
        from mifem.nonlinear import _int_forms
        V = W = functionspace(create_unit_cube(n, jitter=0.2, seed=1), ("P", 1))
        kap, u = Function(V), Function(V)
        kap.x[:], u.x[:] = np.random.default_rng(4).uniform(0.5, 1, (2, V.size))
        a = forms.Form(2, [V, V], [_int_forms(V, V, 2)], [kap, u])
    else:
        R = reference_test_forms(create_unit_cube(n, jitter=0.2, seed=1) if which == "interior"
                                 else create_unit_square(n, n), 1)
        if which == "interior":                              # a discontinuous space not numbered cell by cell
            a = R["matrix"][2]
            V = W = a.function_spaces[0]
            V._dofmap = np.random.default_rng(2).permutation(V.size).astype(np.int32)[V._dofmap]
            R["u_dg"].x[:] = np.random.default_rng(4).uniform(-1, 1, V.size)
        else:
            a = R["matrix"][0]
            V = W = a.function_spaces[0]
    f = cufem.form(a)
    src = f.source()
    kind = "int" if which in ("interior", "facets") else "cell"
    assert "mf_mat_" + kind + "_0" in src and "mf_owner_" not in src
    assert which == "interior" or "mf_ten_" + kind + "_0" in src
    asm = cufem.CUDAAssembler()
    A = asm.create_matrix(f)
    b0 = _some_dofs(V, 0.1, 1)
    b1 = b0 if sets == "equal" and V is W else _some_dofs(W, 0.2, 2)
    none = sets == "none"
    p0 = asm.pack_bcs([] if none else [b0])
    p1 = p0 if b1 is b0 else asm.pack_bcs([] if none else [b1])
    f.to_device()
    asm.pack_coefficients(f)
    o = cpu.OracleAssembler(a) if T is None else None
    rp, cols, _ = A.csr()
    if o is not None:
        orp, ocols, _, _ = o.sparsity()
        assert np.array_equal(rp, orp) and np.array_equal(cols, ocols)
    full = o.assemble_matrix(rp, cols, []) if o is not None else _at_pattern(V, W, rp, cols, T)
    rows = np.repeat(np.arange(V.size), np.diff(rp))
    m0, m1 = np.zeros(V.size, bool), np.zeros(W.size, bool)
    if not none:
        m0[b0.dofs], m1[b1.dofs] = True, True
    for times in (1, 2):
        _lib.check(_lib.lib().mf_assemble_matrix(f.handle, A.handle, p0._get_cpp_bcs(V).handle,
                                                 p1._get_cpp_bcs(W).handle, 2.5, int(times == 1), None))
        asm.synchronize()
        ref = np.where(m0[rows] | m1[cols], 0.0, times * full)
        if V is W:
            ref[(rows == cols) & m0[rows]] = 2.5
        assert _rel(A.csr()[2], ref) <= TOL, times


@pytest.mark.parametrize("which", ["constants", "functions", "vector", "hex", "three", "facets"])
def test_sum_of_forms_with_one_body(which):
    """Two terms with the same element body keep each their constants and
    coefficients."""
    import cudolfinx as cufem
    from mifem.fem import Constant
    print(f"[gpu-test] sum of forms with one body: {which}", flush=True)
    if which == "hex":
        V = functionspace(create_unit_cube(3, "hexahedron", jitter=0.2, seed=1), ("P", 2))
        terms = [forms.hex_source(V, Constant(v)) for v in (1.0, -3.0)]
    else:
        V = functionspace(create_unit_cube(3, jitter=0.2, seed=1), ("P", 2), **({"shape": (3,)} if which == "vector" else {}))
        rng = np.random.default_rng(1)
        if which == "functions":
            fs = [Function(V), Function(V)]
            for f in fs:
                f.x[:] = rng.uniform(-1, 1, V.size)
            terms = [forms.source(V, f) for f in fs]
        elif which == "facets":
            m = V.mesh
            ends = [m.locate_boundary_facets(lambda x, e=e: np.isclose(x[0], e)) for e in (0.0, 1.0)]
            terms = [forms.facet_source(V, Constant(v), e) for v, e in zip((2.0, -5.0), ends)]
        elif which == "vector":
            terms = [forms.source(V, Constant(v)) for v in ([1.0, 2.0, 3.0], [0.5, -7.0, 2.0])]
        else:
            terms = [forms.source(V, Constant(v)) for v in (1.0, -3.0, 5.0)[:3 if which == "three" else 2]]
    L = terms[0]
    for t in terms[1:]:
        L = forms.linear_sum(L, t)
    asm = cufem.CUDAAssembler()
    b = asm.assemble_vector(cufem.form(L))
    asm.synchronize()
    ref = sum(cpu.OracleAssembler(t).assemble_vector() for t in terms)
    assert _rel(b.to_host(), ref) <= TOL


@pytest.mark.parametrize("share", [0.02, 0.3, 1.0])
@pytest.mark.parametrize("which,n", [("heavy", 1), ("heavy", 4), ("light", 3), ("whole", 2), ("facets", 3), ("exterior", 3)])
def test_lifting_by_entity(which, n, share):
    """The per-entity lifting kernel: a body heavy enough for row groups (P2 with 64
    points), light ones, a tensor of more than 256 entries, facets between cells."""
    import dataclasses
    import cudolfinx as cufem
    from mifem.nonlinear import _int_forms, reference_test_forms
    print(f"[gpu-test] lifting by entity: {which} n={n} share={share}", flush=True)
    mesh = create_unit_cube(n, jitter=0.2, seed=1)
    rng = np.random.default_rng(4)
    if which in ("heavy", "exterior"):
        R = reference_test_forms(mesh, 2)
        a = R["matrix"][0 if which == "heavy" else 1]
        R["u"].x[:] = rng.uniform(-1, 1, R["u"].x.size)
    elif which == "facets":
        V = functionspace(mesh, ("P", 1))
        kap, u = Function(V), Function(V)
        kap.x[:], u.x[:] = rng.uniform(0.5, 1, (2, V.size))
        a = forms.Form(2, [V, V], [_int_forms(V, V, 2)], [kap, u])
    else:
        a = _poisson(n, 2)[1] if which == "light" else _elasticity(n)[1]
        a = dataclasses.replace(a, integrals=[dataclasses.replace(a.integrals[0], staged=None)])
    V = a.function_spaces[0]
    bc = _some_dofs(V, share, 6)
    x0 = rng.uniform(-1, 1, V.size)
    f = cufem.form(a)
    kind = {"facets": "int", "exterior": "ext"}.get(which, "cell")
    groups = f.source().split("mf_lift_" + kind + "_0(")[1].split("\n}\n")[0].count("case ")
    assert (groups > 1) == (which == "heavy"), groups
    asm = cufem.CUDAAssembler()
    b = cufem.CUDAVector(asm._ctx, V.size)
    xv = cufem.CUDAVector(asm._ctx, V.size)
    xv.data.upload(x0)
    asm.apply_lifting(b, [f], [asm.pack_bcs([bc])], x0=[xv], scale=0.6)
    asm.synchronize()
    ref = np.zeros(V.size)
    cpu.OracleAssembler(a).apply_lifting(ref, [bc], x0=x0, scale=0.6)
    assert _rel(b.to_host(), ref) <= TOL


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("share", [0.0005, 1.0])
def test_lifting_of_many_heavy_cells(share, noalloc):
    """A heavy body with few and with all of 29 thousand cells to lift: rows in
    groups, and the whole tensor by one thread."""
    import ctypes as C
    import cudolfinx as cufem
    from cudolfinx import _lib
    from mifem.nonlinear import reference_test_forms
    print(f"[gpu-test] lifting of heavy cells: share={share} noalloc={noalloc}", flush=True)
    mesh = create_unit_cube(17, jitter=0.2, seed=1)
    rng = np.random.default_rng(4)
    R = reference_test_forms(mesh, 2)
    a = R["matrix"][0]
    R["u"].x[:] = rng.uniform(-1, 1, R["u"].x.size)
    V = a.function_spaces[0]
    bc = _some_dofs(V, share, 6)
    x0 = rng.uniform(-1, 1, V.size)
    f = cufem.form(a)
    src = f.source()
    most = int(src.split("mf_lift_cell_0(")[1].split("count > ")[1].split(")")[0])
    marked = np.zeros(V.size, bool)
    marked[bc.dofs] = True
    listed = int(marked[V.dofmap].any(axis=1).sum())
    assert (listed > most) == (share == 1.0) and len(V.dofmap) > most, (listed, most)
    asm = cufem.CUDAAssembler()
    b = cufem.CUDAVector(asm._ctx, V.size)
    xv = cufem.CUDAVector(asm._ctx, V.size)
    xv.data.upload(x0)
    dbc = asm.pack_bcs([bc])
    asm.pack_coefficients(f)
    if noalloc:
        _lib.check(_lib.lib().mf_apply_lifting_noalloc(
            (C.c_void_p * 1)(f.handle.value), 1, b.ptr, b.size,
            (C.c_void_p * 1)(dbc._get_cpp_bcs(V).handle.value), (C.c_void_p * 1)(xv.ptr.value), 0.6, None))
    else:
        asm.apply_lifting(b, [f], [dbc], x0=[xv], scale=0.6)
    asm.synchronize()
    ref = np.zeros(V.size)
    cpu.OracleAssembler(a).apply_lifting(ref, [bc], x0=x0, scale=0.6)
    assert _rel(b.to_host(), ref) <= TOL
