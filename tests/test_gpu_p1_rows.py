"""P1 rows by 16 lanes (variant 18, the default on tetrahedra), the default
variants, the lifting and the system call's stored vector, against the oracle."""

import copy

import numpy as np
import pytest

import oracle as O
from dolfinx_amd import fem, graph, la, mesh
from dolfinx_amd._lib import DfxError

from conftest import rel_err
from test_mesh_create import bicone, box_input

pytestmark = pytest.mark.gpu

MESHES = {
    "one": (np.array([[0, 1, 2, 3]]), np.array([[0, 0, 0], [1, 0, 0], [0.2, 1, 0], [0.1, 0.3, 1.]])),
    "box": box_input((5, 3, 4), O.TET, 4),
    "fan": bicone(24),      # 48 cells at a vertex, 27 entries in its row
    "wide": bicone(40),     # 320 contributions to a row, 43 entries
}


@pytest.mark.parametrize("dtype,tol", [(np.float64, 1e-13), (np.float32, 2e-6)])
@pytest.mark.parametrize("name", list(MESHES))
def test_rows_and_lifting(name, dtype, tol):
    cells, x = MESHES[name]
    om = O.Mesh.from_cells(O.TET, cells, x)
    pm = mesh.create_mesh(mesh.CellType.tetrahedron, cells, x)
    V = fem.functionspace(pm, ("Lagrange", 1))
    dm, nd = om.dofmap(1)
    rng = np.random.default_rng(8)
    kap = rng.uniform(0.5, 2.0, (om.num_cells, 1))
    f = rng.standard_normal((om.num_cells, 4))
    a = fem.form("p1_stiffness_reaction", V, kap, [0.7], dtype)
    L = fem.form("p1_source", V, f, None, dtype)
    rp, cols = O.sparsity(dm, dm, nd)
    bdofs = np.nonzero(rng.random(nd) < 0.3)[0].astype(np.int32)
    mark = np.zeros(nd, np.int8)
    mark[bdofs] = 1
    g = rng.standard_normal(nd)
    bc = fem.dirichletbc(V, bdofs, g)
    c = np.array([0.7])
    plain = O.assemble_matrix(O.K_P1TET_A, om.x, om.cells, dm, 1, kap, c, None, None, rp, cols)
    zeroed = O.assemble_matrix(O.K_P1TET_A, om.x, om.cells, dm, 1, kap, c, mark, mark, rp, cols)
    O.set_diagonal(zeroed, bdofs, 1, 2.0, rp, cols)
    for variant in (None, 18):
        if variant is not None:
            a.set_variant(variant)
        A = fem.assemble_matrix(a)
        assert rel_err(A.data, plain) <= tol
        fem.assemble_matrix(a, [], 1.0, A)
        assert rel_err(A.data, 2 * plain) <= tol
        assert rel_err(fem.assemble_matrix(a, [bc], 2.0).data, zeroed) <= tol
    br = O.assemble_vector(O.K_P1TET_L, om.x, om.cells, dm, 1, f, None, nd)
    O.lift_bc(br, O.K_P1TET_A, om.x, om.cells, dm, 1, kap, c, g, mark)
    O.bc_set(br, bdofs, g)
    # a system call from scratch, again over its results, and its parts
    A, b = fem.assemble_system(a, L, [bc], 2.0)
    for _ in range(2):
        assert rel_err(A.data, zeroed) <= tol and rel_err(b.array, br) <= 2 * tol
        fem.assemble_system(a, L, [bc], 2.0, A, b)
    parts = fem.assemble_vector(L)
    fem.apply_lifting(parts, [a], [[bc]])
    fem.set_bc(parts, [bc])
    assert np.array_equal(parts.array, b.array)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("name", list(MESHES))
def test_entries_are_those_of_variant_1(name, dtype):
    """Variant 18 forms and adds the entries in the order and with the
    rounding of the thread-per-row kernel: the same bits."""
    cells, x = MESHES[name]
    V = fem.functionspace(mesh.create_mesh(mesh.CellType.tetrahedron, cells, x), ("Lagrange", 1))
    rng = np.random.default_rng(12)
    kap = rng.uniform(0.5, 2.0, (V.dofmap.list.shape[0], 1))
    a = fem.form("p1_stiffness_reaction", V, kap, [0.7], dtype)
    bdofs = np.nonzero(rng.random(V.num_dofs) < 0.3)[0].astype(np.int32)
    for bcs in ([], [fem.dirichletbc(V, bdofs)]):
        out = []
        for variant in (1, 18):
            a.set_variant(variant)
            A = fem.assemble_matrix(a, bcs)
            fem.assemble_matrix(a, bcs, 1.0, A)  # added to what is there
            out.append(A.data)
        assert np.array_equal(*out)


@pytest.mark.parametrize("cell,n,name", [
    (O.HEX, (6, 5, 4), "q1"), (O.TET, (4, 3, 3), "p3"), (O.TET, (11, 9, 8), "p3")])
def test_defaults_lift_from_the_assemblys_records(cell, n, name):
    """Nonzero data through a system call (the lifting reads the records that
    the matrix assembly left) equals the separate calls, for the variants that
    the library chooses and some others."""
    deg = 3 if name == "p3" else 1
    pm = mesh.create_box([[0, 0, 0], [1, 1, 1]], n, mesh.CellType(cell))
    V = fem.functionspace(pm, ("Lagrange", deg))
    rng = np.random.default_rng(2)
    nc = pm.topology.cells.shape[0]
    a = fem.form(f"{name}_stiffness_reaction", V, rng.uniform(0.5, 2.0, (nc, 1)), [0.3])
    L = (fem.form("q1_source", V, rng.standard_normal((nc, 8))) if name == "q1"
         else fem.form("p3_source", V, None, [1.3]))
    bc = fem.dirichletbc(V, fem.locate_boundary_dofs(V), rng.standard_normal(V.num_dofs))
    ref = None
    for variant in [None] + ([1, 10, 13, 15] if name == "q1" else [3, 7, 16]):
        if variant is not None:
            a.set_variant(variant)
        A, b = fem.assemble_system(a, L, [bc])
        A1 = fem.assemble_matrix(a, [bc])
        b1 = fem.assemble_vector(L)
        fem.apply_lifting(b1, [a], [[bc]])
        fem.set_bc(b1, [bc])
        if variant != 3:  # (LDS atomics: the order of the additions varies)
            assert np.array_equal(A.data, A1.data)
        assert rel_err(b.array, b1.array) <= 1e-14
        ref = ref or (A.data, b.array)
        assert rel_err(A.data, ref[0]) <= 1e-13 and rel_err(b.array, ref[1]) <= 1e-13


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_source_form_of_another_numbering(dtype):
    """A source form whose dofs are numbered otherwise than the stiffness
    form's, on the same geometry: the lifting of a system call goes to the
    stiffness form's rows, as in the separate calls."""
    pm = mesh.create_box([[0, 0, 0], [1, 1, 1]], (5, 4, 3), mesh.CellType.tetrahedron)
    V = fem.functionspace(pm, ("Lagrange", 1))
    rng = np.random.default_rng(6)
    nc = pm.topology.cells.shape[0]
    W = copy.copy(V)
    W._h = None
    W.dofmap = copy.copy(V.dofmap)
    W.dofmap.list = rng.permutation(V.num_dofs).astype(np.int32)[V.dofmap.list]
    a = fem.form("p1_stiffness_reaction", V, rng.uniform(0.5, 2.0, (nc, 1)), [0.7], dtype)
    L = fem.form("p1_source", W, rng.standard_normal((nc, 4)), None, dtype)
    bc = fem.dirichletbc(V, fem.locate_boundary_dofs(V), rng.standard_normal(V.num_dofs))
    parts = fem.assemble_vector(L)
    fem.apply_lifting(parts, [a], [[bc]])
    fem.set_bc(parts, [bc])
    A, b = fem.assemble_system(a, L, [bc])
    for _ in range(2):
        assert np.array_equal(b.array, parts.array)
        fem.assemble_system(a, L, [bc], 1.0, A, b)


@pytest.mark.parametrize("cell,name", [(mesh.CellType.tetrahedron, "p1"),
                                       (mesh.CellType.hexahedron, "q1")])
def test_condition_of_another_space_is_refused(cell, name):
    """Dirichlet data for fewer dofs than the forms have: the system call
    refuses it before any kernel reads it."""
    V, W = (fem.functionspace(mesh.create_box([[0, 0, 0], [1, 1, 1]], n, cell), ("Lagrange", 1))
            for n in ((9, 8, 7), (2, 2, 2)))
    nc, k = V.dofmap.list.shape
    a = fem.form(f"{name}_stiffness_reaction", V, np.ones((nc, 1)), [0.7])
    L = fem.form(f"{name}_source", V, np.ones((nc, k)))
    A, b = fem.assemble_system(a, L)
    small = fem.dirichletbc(W, fem.locate_boundary_dofs(W), np.ones(W.num_dofs))
    with pytest.raises(DfxError, match="BC size does not match"):
        fem.assemble_system(a, L, [small], 1.0, A, b)
    bc = fem.dirichletbc(V, fem.locate_boundary_dofs(V))
    fem.assemble_system(a, L, [bc], 1.0, A, b)
    assert np.array_equal(A.data, fem.assemble_matrix(a, [bc]).data)


@pytest.mark.parametrize("dtype,tol", [(np.float64, 1e-14), (np.float32, 1e-6)])
def test_first_lifting_inside_a_capture(dtype, tol):
    """A P1 form that never lifted can be recorded doing so."""
    V = fem.functionspace(mesh.create_box([[0, 0, 0], [1, 1, 1]], (5, 4, 3),
                                          mesh.CellType.tetrahedron), ("Lagrange", 1))
    rng = np.random.default_rng(9)
    nc, k = V.dofmap.list.shape
    kap, f = rng.uniform(0.5, 2.0, (nc, 1)), rng.standard_normal((nc, k))
    bc = fem.dirichletbc(V, fem.locate_boundary_dofs(V), rng.standard_normal(V.num_dofs))
    x0 = la.Vector.from_array(rng.standard_normal(V.num_dofs).astype(dtype))

    def lifted(a, L, b):
        b.set(0.0)
        fem.assemble_vector(L, b)
        fem.apply_lifting(b, [a], [[bc]], [x0], 0.5)

    L = fem.form("p1_source", V, f, None, dtype)
    ref = la.Vector(V.num_dofs, dtype)
    lifted(fem.form("p1_stiffness_reaction", V, kap, [0.7], dtype), L, ref)
    a, b = fem.form("p1_stiffness_reaction", V, kap, [0.7], dtype), la.Vector(V.num_dofs, dtype)
    g = graph.Graph()
    with g.capture():
        lifted(a, L, b)
    for _ in range(3):
        b.set(7.0)
        g.launch()
        assert rel_err(b.array, ref.array) <= tol
        lifted(a, L, b)  # (its own kernels, eagerly, between the replays)
        assert np.array_equal(b.array, ref.array)


@pytest.mark.parametrize("cell,name", [(mesh.CellType.tetrahedron, "p1"),
                                       (mesh.CellType.hexahedron, "q1")])
def test_first_single_assembly_inside_a_capture(cell, name):
    """A form assembled so far by the batched call alone (which leaves its
    slots, not the plan of the default variant) can be recorded by itself;
    outside of captures it then takes its default variant."""
    V = fem.functionspace(mesh.create_box([[0, 0, 0], [1, 1, 1]], (5, 4, 3), cell),
                          ("Lagrange", 1))
    nc = V.dofmap.list.shape[0]
    kap = np.random.default_rng(4).uniform(0.5, 2.0, (nc, 1))
    bc = fem.dirichletbc(V, fem.locate_boundary_dofs(V))
    a = fem.form(f"{name}_stiffness_reaction", V, kap, [0.7])
    A = fem.create_matrix(a)
    fem.assemble_matrix_batched([a], [bc], [A])
    ref = A.data
    g = graph.Graph()
    with g.capture():
        A.set_value(0.0)
        fem.assemble_matrix(a, [bc], 1.0, A)
    for _ in range(3):
        A.data = np.full(A.nnz, 3.0)
        g.launch()
        assert rel_err(A.data, ref) <= 1e-14
        A.set_value(0.0)
        fem.assemble_matrix(a, [bc], 1.0, A)
        assert rel_err(A.data, ref) <= 1e-14
    a.set_variant(18 if name == "p1" else 15)
    eager = A.data
    A.set_value(0.0)
    fem.assemble_matrix(a, [bc], 1.0, A)
    assert np.array_equal(A.data, eager)
