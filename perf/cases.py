"""Workloads of the assemble-and-solve path: what a program using dolfinx_amd
has it do, each through the package's public entry points.

  system  A and b of one boundary value problem re-assembled into a matrix and
          a vector that exist already (a new time step or coefficient):
          fem.assemble_system with Dirichlet rows, lifting and set_bc.
  spmv    y = A x with an assembled matrix (MatrixCSR.mult).
  cg      Jacobi-CG to a tolerance from x = 0 (solvers.cg).
  mixed   the same solve by FP32 Jacobi-CG inside FP64 refinement
          (solvers.mixed_refinement).
  serve   requests that bring their own coefficients and wait for their
          solution (serve.SolveService.run): packing, batched assembly,
          right-hand sides, the batched CG and the solutions on the host.

Spaces: p1 and p3 (scalar, tetrahedra), q1 (scalar, hexahedra), p2 (vector
elasticity, tetrahedra), on boxes of nx x ny x nz cubes. Coefficients follow
the package's own problems: kappa log-normal per cell (p1, q1), U[1, 10] (p3),
Young's modulus U[0.5, 2] (p2).

The host part that does not depend on the seed (mesh, dofmap, sparsity
pattern, serving templates) is set up once per size and kept, as a program
that solves on one mesh repeatedly keeps it.
"""

from __future__ import annotations

import ctypes
from collections import OrderedDict

import numpy as np
import torch

from dolfinx_amd import _lib, fem, la, mesh, serve, solvers

# space -> (cell, degree, block size, bilinear form, linear form)
SPACES = {
    "p1": (mesh.CellType.tetrahedron, 1, 1, "p1_stiffness_reaction", "p1_source"),
    "q1": (mesh.CellType.hexahedron, 1, 1, "q1_stiffness_reaction", "q1_source"),
    "p2": (mesh.CellType.tetrahedron, 2, 3, "p2_elasticity", "p2_body_force"),
    "p3": (mesh.CellType.tetrahedron, 3, 1, "p3_stiffness_reaction", "p3_source"),
}
NU = 0.3  # Poisson ratio of the elasticity problems


def _case(kind, space, nx, ny, nz, dtype="f64", g=False, tuned=False, rtol=0.0, name=None):
    c = {"kind": kind, "space": space, "nx": nx, "ny": ny, "nz": nz, "dtype": dtype, "g": g,
         "tuned": tuned, "rtol": rtol}
    return c if name is None else {"name": name, **c}


def listed():
    return [
        # the smallest re-assembly: a coarse mesh in a parameter study, where
        # launches and host calls are the whole cost
        _case("system", "p1", 9, 8, 7, name="p1_system_9x8x7"),
        # FP32 assembly on an odd box, nonzero Dirichlet data (so lifting works)
        _case("system", "p1", 61, 47, 53, dtype="f32", g=True, name="p1_system_61x47x53_f32"),
        # the benchmark's headline step: Q1, 128^3 hexahedra, tuned as it does
        _case("system", "q1", 128, 128, 128, tuned=True, name="q1_system_128"),
        # vector elasticity at the size of the elasticity configuration
        _case("system", "p2", 48, 48, 48, name="p2_system_48"),
        # the high-order configuration
        _case("system", "p3", 24, 24, 24, tuned=True, name="p3_system_24"),
        # one matrix-vector product of a caller's own Krylov method
        _case("spmv", "q1", 128, 128, 128, name="q1_spmv_128"),
        # the small Poisson configuration's solve
        _case("cg", "p1", 32, 32, 32, rtol=1e-10, name="p1_cg_32"),
        # the precision configuration's FP64 solve, and a mixed one on a ragged box
        _case("cg", "q1", 128, 128, 128, rtol=1e-8, name="q1_cg_128"),
        _case("mixed", "q1", 96, 80, 111, rtol=1e-8, name="q1_mixed_96x80x111"),
        # elasticity on a ragged box, and the high-order solve
        _case("cg", "p2", 24, 19, 17, rtol=1e-8, name="p2_cg_24x19x17"),
        _case("cg", "p3", 24, 24, 24, rtol=1e-8, name="p3_cg_24"),
        # sixteen requests at once over the serving range of meshes
        {"name": "serve_16", "kind": "serve", "lo": 8, "hi": 48, "requests": 16},
    ]


def draw(rng):
    kind = rng.choice(["system"] * 5 + ["spmv"] * 2 + ["cg"] * 3 + ["mixed", "serve"])
    if kind == "serve":
        lo = rng.randint(8, 20)
        return {"kind": "serve", "lo": lo, "hi": rng.randint(lo + 4, 47),
                "requests": rng.randint(1, 15)}
    space = rng.choice(["p1", "q1", "p2", "p3"]) if kind != "mixed" else rng.choice(["p1", "q1"])
    top = {("system", "p1"): 56, ("system", "q1"): 116, ("system", "p2"): 36, ("system", "p3"): 22,
           ("spmv", "p1"): 56, ("spmv", "q1"): 116, ("spmv", "p2"): 28, ("spmv", "p3"): 22,
           ("cg", "p1"): 56, ("cg", "q1"): 96, ("cg", "p2"): 16, ("cg", "p3"): 18,
           ("mixed", "p1"): 52, ("mixed", "q1"): 84}[kind, space]
    n = 4.0 * (top / 4.0) ** rng.random()
    n = [max(3, round(n * rng.uniform(0.8, 1.25))) for _ in range(3)]
    while n[0] * n[1] * n[2] > top ** 3:
        n[n.index(max(n))] -= 1
    solve = kind in ("cg", "mixed")
    return _case(kind, space, *n, dtype="f64" if solve else rng.choice(["f64", "f64", "f32"]),
                 g=rng.random() < 0.5, tuned=kind in ("system", "spmv") and rng.random() < 0.5,
                 rtol=rng.choice([1e-6, 1e-8, 1e-10]) if solve else 0.0)


# ---------------------------------------------------------------------------
# Host setup and inputs
# ---------------------------------------------------------------------------

class _Setup:
    """Mesh, space, Dirichlet dofs and sparsity pattern of one box."""

    def __init__(self, space, n):
        cell, degree, bs, _, _ = SPACES[space]
        self.mesh = mesh.create_box([[0.0, 0.0, 0.0], [1.0, 1.0, 1.0]], n, cell)
        self.V = fem.functionspace(self.mesh, ("Lagrange", degree, (3,) if bs == 3 else None))
        # elasticity: the face x = 0 is clamped; else the whole boundary
        self.dofs = (fem.locate_boundary_dofs(self.V, axis=0, value=0.0) if space == "p2"
                     else fem.locate_boundary_dofs(self.V))
        h = ctypes.c_void_p()
        _lib.call("dfx_sparsity_create", self.V.handle, self.V.handle, ctypes.byref(h))
        self.pattern = fem.SparsityPattern(h)


_kept: OrderedDict = OrderedDict()


def _keep(key, make, most=6):
    if key in _kept:
        _kept.move_to_end(key)
    else:
        _kept[key] = make()
        while len(_kept) > most:
            _kept.popitem(last=False)
    return _kept[key]


def _setup(case):
    n = (case["nx"], case["ny"], case["nz"])
    return _keep((case["space"], n), lambda: _Setup(case["space"], n))


def _service(case):
    return _keep(("serve", case["lo"], case["hi"], case["requests"]),
                 lambda: serve.SolveService(sizes=sorted(set(_sizes(case)))))


def _sizes(case):
    """Mesh sizes of the requests, spread evenly over lo..hi."""
    lo, hi, r = case["lo"], case["hi"], case["requests"]
    return [lo + (hi - lo) * i // max(1, r - 1) for i in range(r)]


def _fields(case, seed):
    """Coefficients of the seed, by input cell and vertex: packed coefficients
    of both forms, their constants and the Dirichlet values by dof."""
    S = _setup(case)
    rng = np.random.Generator(np.random.PCG64(seed))
    nc, nv = S.mesh.topology.cells.shape[0], S.mesh.geometry.x.shape[0]
    if case["space"] == "p2":
        E = rng.uniform(0.5, 2.0, nc)
        lam, mu = E * NU / ((1 + NU) * (1 - 2 * NU)), E / (2 * (1 + NU))
        wa, ca = fem.pack_cellwise(S.mesh, np.stack([lam, mu], 1)), None
        wl, cl = None, [0.1 * rng.standard_normal(), 0.0, -1.0]
    elif case["space"] == "p3":
        wa, ca = fem.pack_cellwise(S.mesh, rng.uniform(1.0, 10.0, nc)), [1.0]
        wl, cl = None, [rng.uniform(0.5, 2.0)]
    else:
        wa = fem.pack_cellwise(S.mesh, np.exp(rng.standard_normal(nc)))
        ca = [rng.uniform(0.0, 10.0)]
        wl, cl = fem.pack_vertexwise(S.mesh, 1.0 + 0.2 * rng.standard_normal(nv)), None
    g = 1.0 + 0.1 * rng.standard_normal(S.V.num_dofs) if case["g"] else None
    return wa, ca, wl, cl, g


def _dtype(case):
    return np.float64 if case["dtype"] == "f64" else np.float32


class _View:
    """Device buffer of a Vector (values at byte 8 of its handle) or a
    MatrixCSR (byte 56) for torch, which shares and does not copy it; the
    owner is kept alive. A C++ program linked with the library hands the same
    pointers on."""

    def __init__(self, owner, n, offset):
        self.owner = owner
        address = ctypes.c_void_p.from_address(owner.handle.value + offset).value
        self.__cuda_array_interface__ = {
            "shape": (int(n),), "typestr": np.dtype(owner.dtype).str, "data": (address, False),
            "strides": None, "version": 2}


def _vector(v):
    return torch.as_tensor(_View(v, v.size, 8), device="cuda")


def _values(A):
    return torch.as_tensor(_View(A, A.nnz * A.bs * A.bs, 56), device="cuda")


def _requests(case, seed):
    out = []
    for i, n in enumerate(_sizes(case)):
        rng = np.random.Generator(np.random.PCG64([seed, i]))
        out.append(serve.Request(i, n, np.exp(0.5 * rng.standard_normal(6 * n ** 3)),
                                 float(rng.uniform(0.0, 10.0)), rng.standard_normal((n + 1) ** 3)))
    return out


def _problem(case, S, fields, dtype):
    """Forms, condition, matrix and right-hand side, assembled once (so the
    forms hold their plans for the pattern)."""
    wa, ca, wl, cl, g = fields
    fa, fl = SPACES[case["space"]][3:]
    a = fem.form(fa, S.V, wa, ca, dtype)
    L = fem.form(fl, S.V, wl, cl, dtype)
    bc = fem.dirichletbc(S.V, S.dofs, g)
    A = la.MatrixCSR.from_sparsity(S.pattern, dtype)
    b = la.Vector(S.V.num_dofs, dtype)
    if case["tuned"]:
        a.autotune(A, bc)
    fem.assemble_system(a, L, [bc], 1.0, A, b)
    return a, L, bc, A, b


def prepare(case, seed):
    if case["kind"] == "serve":
        return {"kind": "serve", "service": _service(case), "requests": _requests(case, seed)}
    S = _setup(case)
    fields = _fields(case, seed)
    a, L, bc, A, b = _problem(case, S, fields, _dtype(case))
    s = {"kind": case["kind"], "A": A, "b": b, "rtol": case["rtol"], "outA": _values(A),
         "outb": _vector(b)}
    if case["kind"] == "system":
        s.update(a=a, L=L, bc=bc)
        return s
    x = la.Vector(S.V.num_dofs, _dtype(case))
    s.update(x=x, outx=_vector(x))
    if case["kind"] == "spmv":
        if case["tuned"]:
            A.autotune()
        x.array = _spmv_x(case, seed, x.size)
        s["y"] = la.Vector(S.V.num_dofs, _dtype(case))
        s["outy"] = _vector(s["y"])
    elif case["kind"] == "mixed":
        s["A32"] = _problem(case, S, fields, np.float32)[3]
    return s


def _spmv_x(case, seed, n):
    x = np.random.Generator(np.random.PCG64([seed, 1])).standard_normal(n)
    return x.astype(_dtype(case))


def run(state):
    kind = state["kind"]
    if kind == "system":
        fem.assemble_system(state["a"], state["L"], [state["bc"]], 1.0, state["A"], state["b"])
        return {"A": state["outA"], "b": state["outb"]}
    if kind == "spmv":
        state["y"].set(0.0)
        state["A"].mult(state["x"], state["y"])
        return {"y": state["outy"]}
    if kind == "cg":
        state["x"].set(0.0)
        solvers.cg(state["A"], state["b"], state["x"], rtol=state["rtol"], max_it=50000)
        return {"x": state["outx"]}
    if kind == "mixed":
        state["x"].set(0.0)
        solvers.mixed_refinement(state["A"], state["A32"], state["b"], state["x"],
                                 rtol=state["rtol"])
        return {"x": state["outx"]}
    reqs = state["requests"]
    state["service"].run(reqs, rate=1e6, keep_solutions=[r.rid for r in reqs])
    return [r.x for r in reqs]


# ---------------------------------------------------------------------------
# Work and tolerance
# ---------------------------------------------------------------------------

# CG iterations per cube along the longest side, as this path's problems take
# them at a reduction of 1e-8 (one more power of ten: an eighth more)
ITERATIONS = {"p1": 4.1, "q1": 2.55, "p2": 48.0, "p3": 19.2}
# operations of one cell's element matrix and vector
CELL_FLOPS = {"p1": 300.0, "q1": 1200.0, "p2": 10.0 * 10.0 * 80.0, "p3": 20.0 * 20.0 * 14.0}


def _cg_work(space, nnz, N, n, rtol, s):
    its = ITERATIONS[space] * n * (1.0 - 0.125 * (8.0 + np.log10(rtol)))
    bs = SPACES[space][2]
    per = nnz * (s + 4.0 / (bs * bs)) + 8.0 * N * s  # matrix once, vectors of a fused iteration
    return its * per, its * (2.0 * nnz + 12.0 * N)


def work(case):
    if case["kind"] == "serve":
        nbytes = flops = 0.0
        for n in _sizes(case):
            N, edges = (n + 1) ** 3, 3 * n * (n + 1) ** 2 + 3 * n * n * (n + 1) + n ** 3
            nnz, cells = N + 2 * edges, 6 * n ** 3
            w = _cg_work("p1", nnz, N, n, 1e-8, 8)
            nbytes += w[0] + cells * 24.0 + N * 48.0 + nnz * 8.0
            flops += w[1] + cells * CELL_FLOPS["p1"]
        return {"bytes": nbytes, "flops": flops}
    S = _setup(case)
    bs = SPACES[case["space"]][2]
    blocks = S.pattern.num_nonzeros
    nnz, N = blocks * bs * bs, S.V.num_dofs
    s = 8 if case["dtype"] == "f64" else 4
    cells, k = S.V.dofmap.list.shape
    if case["kind"] == "system":
        coeffs = {"p1": 5, "q1": 9, "p2": 2, "p3": 1}[case["space"]]
        nbytes = (cells * (4.0 * k + coeffs * s) + S.mesh.geometry.x.shape[0] * 3.0 * s
                  + nnz * s + N * s)
        return {"bytes": nbytes, "flops": cells * CELL_FLOPS[case["space"]]}
    if case["kind"] == "spmv":
        return {"bytes": nnz * s + blocks * 4.0 + N / bs * 4.0 + 2.0 * N * s, "flops": 2.0 * nnz}
    if case["kind"] == "mixed":
        s = 4
    w = _cg_work(case["space"], nnz, N, max(case["nx"], case["ny"], case["nz"]), case["rtol"], s)
    return {"bytes": w[0], "flops": w[1]}


# Relative errors against exact(), measured on MI355X over the spaces: FP64
# systems and products 1.2e-16..3.3e-16 (p1, q1), 7e-16..1.1e-15 (p2) and
# 4e-15..7.4e-15 (p3, its reference tensors), FP32 ones 2.2e-7..4.1e-7; four
# times those. A solve to rtol was 0.05 to 0.09 rtol off where the tolerance
# is 1e-6 and 1e-8, served solutions (random loads) up to 2.9e-8.
ROUNDING = {"p1": 1.5e-15, "q1": 1.5e-15, "p2": 5e-15, "p3": 3e-14}


def tolerance(case):
    if case["kind"] == "serve":
        return {"rel": 1e-7}
    if case["kind"] in ("cg", "mixed"):
        return {"rel": 0.4 * case["rtol"]}
    return {"rel": ROUNDING[case["space"]] if case["dtype"] == "f64" else 1.6e-6}


# ---------------------------------------------------------------------------
# The same results in 64 bits with plain torch (the mesh's numbering, dofmap
# and pattern are inputs: they fix the order of the results)
# ---------------------------------------------------------------------------

def _tet_nodes(degree):
    v = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]], float)
    edges = [(2, 3), (1, 3), (1, 2), (0, 3), (0, 2), (0, 1)]
    t = {1: [], 2: [0.5], 3: [0.5 - 0.5 / np.sqrt(5.0), 0.5 + 0.5 / np.sqrt(5.0)]}[degree]
    nodes = list(v) + [v[a] + s * (v[b] - v[a]) for a, b in edges for s in t]
    if degree == 3:
        nodes += [(v[a] + v[b] + v[c]) / 3
                  for a, b, c in [(1, 2, 3), (0, 2, 3), (0, 1, 3), (0, 1, 2)]]
    return np.array(nodes)


def _reference(space):
    """Stiffness products S[a, b, i, j] = int d_a phi_i d_b phi_j and mass
    M[i, j] on the reference cell, by Gauss points of sufficient degree."""
    p, w = np.polynomial.legendre.leggauss(6)
    p, w = 0.5 + 0.5 * p, 0.5 * w
    u, v, z = (q.ravel() for q in np.meshgrid(p, p, p, indexing="ij"))
    wt = (w[:, None, None] * w[None, :, None] * w[None, None, :]).ravel()
    if space == "q1":
        X = np.stack([u, v, z], 1)
        nodes = np.array([[i & 1, i >> 1 & 1, i >> 2] for i in range(8)], float)
        powers = [(i & 1, i >> 1 & 1, i >> 2) for i in range(8)]
    else:
        degree = SPACES[space][1]
        X = np.stack([u, v * (1 - u), z * (1 - u) * (1 - v)], 1)
        wt = wt * (1 - u) ** 2 * (1 - v)
        nodes = _tet_nodes(degree)
        powers = [(i, j, l) for i in range(degree + 1) for j in range(degree + 1 - i)
                  for l in range(degree + 1 - i - j)]

    def values(Y, d=None):
        cols = []
        for e in powers:
            c = np.ones(len(Y))
            for a in range(3):
                if a == d:
                    c = c * (e[a] * Y[:, a] ** (e[a] - 1) if e[a] else 0.0)
                else:
                    c = c * Y[:, a] ** e[a]
            cols.append(c)
        return np.stack(cols, 1)

    B = np.linalg.inv(values(nodes))
    D = [values(X, a) @ B for a in range(3)]
    P = values(X) @ B
    S = np.array([[(D[a] * wt[:, None]).T @ D[b] for b in range(3)] for a in range(3)])
    return S, (P * wt[:, None]).T @ P


def _exact_system(S, space, fields):
    """(values, b, row of each value's block, device) of the problem."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    t = lambda v: torch.as_tensor(np.ascontiguousarray(v), device=dev)  # noqa: E731
    wa, ca, wl, cl, g = fields
    bs = SPACES[space][2]
    RS, RM = (t(r) for r in _reference(space))
    x, cells, dofs = t(S.mesh.geometry.x), t(S.mesh.geometry.dofmap).long(), t(S.V.dofmap.list).long()
    k, N = dofs.shape[1], S.V.num_dofs
    rp, cols = t(S.pattern.row_ptr), t(S.pattern.cols).long()
    nb = len(S.pattern.row_ptr) - 1
    rows = torch.repeat_interleave(torch.arange(nb, device=dev), rp[1:] - rp[:-1])
    keys = rows * nb + cols
    vals = torch.zeros(len(cols) * bs * bs, dtype=torch.float64, device=dev)
    b = torch.zeros(N, dtype=torch.float64, device=dev)
    fixed = torch.zeros(N, dtype=torch.float64, device=dev)
    fixed[t(S.dofs).long()] = 1.0
    gv = torch.zeros(N, dtype=torch.float64, device=dev) if g is None else t(g)
    waT = t(wa)
    wlT = None if wl is None else t(wl)
    corner = [1, 2, 4] if space == "q1" else [1, 2, 3]
    comp = torch.arange(bs, device=dev)
    step = 150_000 if k <= 8 else 20_000
    for lo in range(0, len(cells), step):
        c = cells[lo:lo + step]
        d = dofs[lo:lo + step]
        X = x[c]
        J = torch.stack([X[:, q] - X[:, 0] for q in corner], 2)
        det = torch.linalg.det(J).abs()
        Ji = torch.linalg.inv(J)
        w = waT[lo:lo + step]
        n = len(c)
        if bs == 1:
            G = (Ji @ Ji.transpose(1, 2).contiguous()) * (w[:, 0] * det)[:, None, None]
            E = (G.reshape(n, 9) @ RS.reshape(9, k * k)) + (ca[0] * det)[:, None] * RM.reshape(1, -1)
            E = E.reshape(n, k, k)
            f = wlT[lo:lo + step] if wlT is not None else torch.full((n, k), float(cl[0]),
                                                                     dtype=torch.float64, device=dev)
            e = (f @ RM) * det[:, None]
            u = d
        else:
            # D[c, a, b, i, j] = int d_a phi_i d_b phi_j on the cell
            D = torch.einsum("cra,rsij->caisj", Ji, RS).reshape(n, 3 * k, 3, k)
            D = torch.einsum("cmsj,csb->cmbj", D, Ji).reshape(n, 3, k, 3, k)
            D = D.permute(0, 1, 3, 2, 4) * det[:, None, None, None, None]
            lam, mu = w[:, 0, None, None], w[:, 1, None, None]
            tr = D[:, 0, 0] + D[:, 1, 1] + D[:, 2, 2]
            E = torch.empty(n, k, 3, k, 3, dtype=torch.float64, device=dev)
            for a in range(3):
                for q in range(3):
                    E[:, :, a, :, q] = lam * D[:, a, q] + mu * D[:, q, a] + (mu * tr if a == q else 0)
            E = E.reshape(n, 3 * k, 3 * k)
            load = torch.tensor([float(v) for v in cl], dtype=torch.float64, device=dev)
            e = ((RM.sum(1)[None, :] * det[:, None])[:, :, None] * load).reshape(n, 3 * k)
            u = (d[:, :, None] * 3 + comp).reshape(n, 3 * k)
        m = fixed[u]
        e = e - (E @ (m * gv[u])[:, :, None])[:, :, 0]
        b.index_add_(0, u.reshape(-1), e.reshape(-1))
        E = E * (1 - m)[:, :, None] * (1 - m)[:, None, :]
        pos = torch.searchsorted(keys, (d[:, :, None] * nb + d[:, None, :]).reshape(-1))
        if bs == 3:
            pos = pos.reshape(n, k, 1, k, 1) * 9 + comp[:, None, None] * 3 + comp
        vals.index_add_(0, pos.reshape(-1), E.reshape(-1))
    on = torch.nonzero(fixed)[:, 0]
    at = torch.searchsorted(keys, (on // bs) * (nb + 1))
    vals[at * bs * bs + (on % bs) * (bs + 1)] = 1.0
    b[on] = gv[on]
    return vals, b, rows, cols


def _scalar(vals, rows, cols, bs):
    """Scalar (row, column) of every value of a block matrix."""
    if bs == 1:
        return rows, cols
    i = torch.arange(bs, device=rows.device)
    r = (rows[:, None, None] * bs + i[:, None]).expand(-1, bs, bs).reshape(-1)
    c = (cols[:, None, None] * bs + i).expand(-1, bs, bs).reshape(-1)
    return r, c


def _solve(vals, b, rows, cols):
    """Jacobi-CG far past the tolerance of the cases."""
    def mult(p):
        return torch.zeros_like(b).index_add_(0, rows, vals * p[cols])

    diag = torch.zeros_like(b).index_add_(0, rows, torch.where(rows == cols, vals, 0.0))
    x, r = torch.zeros_like(b), b.clone()
    z = r / diag
    p, rz, stop = z.clone(), torch.dot(r, z), 1e-26 * torch.dot(b, b)
    for it in range(20000):
        q = mult(p)
        alpha = rz / torch.dot(p, q)
        x += alpha * p
        r -= alpha * q
        z = r / diag
        new = torch.dot(r, z)
        p = z + (new / rz) * p
        rz = new
        if it % 32 == 31 and torch.dot(r, r) < stop:
            break
    return x


def exact(case, seed):
    if case["kind"] == "serve":
        out = []
        for r in _requests(case, seed):
            S = _keep(("p1", (r.n,) * 3), lambda: _Setup("p1", (r.n,) * 3), most=64)
            fields = (fem.pack_cellwise(S.mesh, r.kappa), [r.c],
                      fem.pack_vertexwise(S.mesh, r.f), None, None)
            vals, b, rows, cols = _exact_system(S, "p1", fields)
            out.append(_solve(vals, b, rows, cols).cpu().numpy())
        return out
    S = _setup(case)
    vals, b, rows, cols = _exact_system(S, case["space"], _fields(case, seed))
    if case["kind"] == "system":
        return {"A": vals, "b": b}
    rows, cols = _scalar(vals, rows, cols, SPACES[case["space"]][2])
    if case["kind"] == "spmv":
        x = torch.as_tensor(_spmv_x(case, seed, len(b)), device=vals.device).double()
        return {"y": torch.zeros_like(b).index_add_(0, rows, vals * x[cols])}
    return {"x": _solve(vals, b, rows, cols)}
