"""Measured cases: what a program built on this package has the GPU do.

Seven operations over the sizes of this repository's benchmarks and tests (2D
grids of 16 to 1024 cells a side, tetrahedral meshes of 6 to 128, degrees 1 to
4, FP64 and FP32):

  matrix      BilinearForm.assembly of diffusion (+ mass) into a CSR matrix
  vector      LinearForm.assembly of a source
  elasticity  BilinearForm.assembly of linear elasticity on a vector space
  element     element matrices on the matrix cores (method='mfma_*')
  dirichlet   DirichletBC.apply on an assembled matrix and right-hand side
  spmv        A @ x with an assembled matrix
  solve       a whole step: assemble, boundary condition, multigrid setup,
              preconditioned CG (or FP32 corrections with FP64 residuals)

A case holds: op; dim; nx, ny, nz (nz 0 in 2D); mesh ('box': from_box, 'free':
the same box triangulated with moved nodes and shuffled numbering, given as
node and cell arrays); p; q (quadrature index, 0: the default); dtype; coef;
mass; form.
"""
import math

import numpy as np
import torch

import fealpy_amd as fa
from fealpy_amd import expr
from fealpy_amd.fem.pattern import pattern_of
from fealpy_amd.solver import GeometricMG
from fealpy_amd.solver.refine import cg_refine

PI = math.pi
DTYPES = {"f64": torch.float64, "f32": torch.float32}


def _case(op, dims, p, *, mesh="box", q=0, dtype="f64", coef="cell", mass=False, form="", name=None):
    c = {"op": op, "dim": len(dims), "nx": dims[0], "ny": dims[1], "nz": dims[2] if len(dims) == 3 else 0,
         "mesh": mesh, "p": p, "q": q, "dtype": dtype, "coef": coef, "mass": mass, "form": form}
    return c if name is None else {"name": name, **c}


def listed():
    return [
        # one request of the solve service: a small 2D problem, where launches and latency count
        _case("solve", (64, 64), 1, form="cg", name="solve_tri_p1_64"),
        # the headline workload: 2.1M DOFs, FP64 system solved by FP32 corrections
        _case("solve", (128, 128, 128), 1, q=2, form="refine", name="solve_tet_p1_128"),
        # its parts that every time step or coefficient update repeats
        _case("matrix", (128, 128, 128), 1, q=2, name="matrix_tet_p1_128"),
        _case("vector", (128, 128, 128), 1, q=2, coef="cellexpr", name="vector_tet_p1_128"),
        # a mesh from a file: nothing known about its numbering, ragged size, diffusion + reaction
        _case("matrix", (71, 83, 64), 1, mesh="free", mass=True, name="matrix_free_p1_71"),
        # second order in 2D at an ordinary size
        _case("matrix", (192, 192), 2, name="matrix_tri_p2_192"),
        # third order in 3D, coefficient and source given as functions of the point
        _case("matrix", (48, 48, 48), 3, q=5, coef="expr", mass=True, name="matrix_tet_p3_48"),
        _case("vector", (48, 48, 48), 3, q=5, coef="expr", name="vector_tet_p3_48"),
        # displacement unknowns of a clamped block
        _case("elasticity", (40, 40, 40), 2, q=5, name="elasticity_tet_p2_40"),
        # fourth-order element matrices on the matrix cores, 16-bit inputs chosen by the caller
        _case("element", (48, 48, 48), 4, q=6, dtype="bf16", coef="point", mass=True, name="element_tet_p4_48"),
        # the boundary condition of a ragged box
        _case("dirichlet", (100, 113, 90), 1, q=2, name="dirichlet_tet_p1_100"),
        # the operator of a user's own iteration
        _case("spmv", (48, 45, 50), 2, name="spmv_tet_p2_48"),
    ]


def _cells(c):
    return 6 * c["nx"] * c["ny"] * c["nz"] if c["dim"] == 3 else 2 * c["nx"] * c["ny"]


def _ldof(c):
    return math.comb(c["p"] + c["dim"], c["dim"])


def draw(rng):
    op = rng.choice(["matrix", "matrix", "vector", "vector", "elasticity", "element", "dirichlet", "spmv", "solve"])

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    while True:
        dim = 3 if op == "element" else rng.choice((2, 3))
        p = rng.choice((1, 2, 3, 4))
        mesh = "box"
        q, dtype, coef, mass, form = 0, "f64", "cell", False, ""
        lo, hi = (16, 1024) if dim == 2 else (6, 128)
        if op == "solve":
            p = rng.choice((1, 2)) if dim == 2 else 1
            hi = 512 if dim == 2 else 128
            form = rng.choice(("cg", "refine"))
        elif op == "matrix":
            mesh = rng.choice(("box", "free"))
            coef = rng.choice(("cell", "expr", "point"))
            mass = rng.random() < 0.5
            dtype = rng.choice(("f64", "f64", "f32"))
        elif op == "vector":
            mesh = rng.choice(("box", "free"))
            coef = rng.choice(("cell", "expr", "cellexpr", "point"))
        elif op == "elasticity":
            p = rng.choice((1, 2, 3))
            mesh = rng.choice(("box", "free"))
        elif op == "element":
            p = rng.choice((2, 3, 4))
            q, dtype, coef, mass = p + 2, rng.choice(("bf16", "fp32")), "point", True
            hi = 48
        else:
            p = rng.choice((1, 2))
            mesh = rng.choice(("box", "free"))
            dtype = rng.choice(("f64", "f32")) if op == "spmv" else "f64"
        n = log_int(lo, hi)
        dims = tuple(min(hi, max(lo, int(round(n * rng.uniform(0.8, 1.25))))) for _ in range(dim))
        if op == "solve" and rng.random() < 0.5:
            dims = (n,) * dim
        c = _case(op, dims, p, mesh=mesh, q=q, dtype=dtype, coef=coef, mass=mass, form=form)
        ncomp = dim if op == "elasticity" else 1
        entries = _cells(c) * (ncomp * _ldof(c)) ** 2
        points = _cells(c) * (p + 3) ** dim                     # bounds the quadrature work
        if op == "solve" and _cells(c) <= 6 * 128 ** 3 or op == "element" and entries <= 4e8 \
                or op in ("matrix", "elasticity") and entries <= 1.5e8 and (coef == "cell" or points <= 2.5e7) \
                or op == "vector" and points <= 6e7 or op in ("dirichlet", "spmv") and entries <= 1e8:
            return c


# ---- inputs ------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _shuffled_in_windows(n, window, g):
    """A permutation of n that moves every index within a window (file meshes are ordered roughly by place)."""
    key = torch.arange(n, device="cuda") // window + torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
    return torch.argsort(key)


def _mesh(c, g):
    dims = (c["nx"], c["ny"], c["nz"])[:c["dim"]]
    kw = dict(zip(("nx", "ny", "nz"), dims), device=torch.device("cuda"))
    cls = fa.TetrahedronMesh if c["dim"] == 3 else fa.TriangleMesh
    mesh = cls.from_box(**kw)
    if c["mesh"] == "box":
        return mesh
    node, cell = mesh.node, mesh.cell.long()
    h = torch.tensor([1.0 / n for n in dims], dtype=torch.float64, device="cuda")
    inside = ((node > 1e-9) & (node < 1 - 1e-9)).all(dim=1, keepdim=True)
    node = node + inside * h * (0.2 * torch.rand(node.shape, generator=g, device="cuda", dtype=torch.float64) - 0.1)
    perm = _shuffled_in_windows(node.shape[0], 512, g)
    new = torch.empty_like(perm)
    new[perm] = torch.arange(perm.shape[0], device="cuda")
    cell = new[cell][_shuffled_in_windows(cell.shape[0], 2048, g)]
    return cls(node[perm].contiguous(), cell.to(torch.int32).contiguous())


def _amplitudes(seed):
    """(a, 8 Fourier modes (amplitude, kx, ky)) of the seed's functions."""
    r = np.random.default_rng(seed)
    a = float(r.uniform(0.3, 0.7))
    modes = [(float(r.standard_normal()), int(r.integers(1, 9)), int(r.integers(1, 9))) for _ in range(8)]
    return a, modes


def _lognormal(nc, g):
    return torch.exp(torch.randn(nc, generator=g, device="cuda", dtype=torch.float64))


def _quadrature(c):
    return c["q"] or c["p"] + 3


def _sines(dim):
    x, y, z = expr.x, expr.y, expr.z
    u = expr.sin(PI * x) * expr.sin(PI * y)
    return u * expr.sin(PI * z) if dim == 3 else u


def _diffusion_expr(dim, a):
    x, y, z = expr.x, expr.y, expr.z
    t = a * expr.sin(2 * PI * x) * expr.cos(2 * PI * y)
    return 1 + (t * z if dim == 3 else t)


def _diffusion_at(pts, a):
    t = a * torch.sin(2 * PI * pts[..., 0]) * torch.cos(2 * PI * pts[..., 1])
    return 1 + (t * pts[..., 2] if pts.shape[-1] == 3 else t)


def _source_expr(dim, a, modes):
    """3D: -div(k grad u) + u of the smooth k and u = sin sin sin; 2D: the Fourier modes of a service request."""
    x, y, z = expr.x, expr.y, expr.z
    sin, cos = expr.sin, expr.cos
    if dim == 2:
        f = None
        for m, kx, ky in modes:
            t = m * sin(kx * PI * x) * sin(ky * PI * y)
            f = t if f is None else f + t
        return f
    k, u = _diffusion_expr(3, a), _sines(3)
    dk = (2 * PI * a * cos(2 * PI * x) * cos(2 * PI * y) * z, -2 * PI * a * sin(2 * PI * x) * sin(2 * PI * y) * z,
          a * sin(2 * PI * x) * cos(2 * PI * y))
    du = (PI * cos(PI * x) * sin(PI * y) * sin(PI * z), PI * sin(PI * x) * cos(PI * y) * sin(PI * z),
          PI * sin(PI * x) * sin(PI * y) * cos(PI * z))
    return 3 * PI ** 2 * k * u - (dk[0] * du[0] + dk[1] * du[1] + dk[2] * du[2]) + u


def _source_at(pts, a, modes):
    s, co = torch.sin(PI * pts), torch.cos(PI * pts)
    if pts.shape[-1] == 2:
        return sum(m * torch.sin(kx * PI * pts[..., 0]) * torch.sin(ky * PI * pts[..., 1]) for m, kx, ky in modes)
    s2, c2, z = torch.sin(2 * PI * pts), torch.cos(2 * PI * pts), pts[..., 2]
    u = s.prod(dim=-1)
    k = 1 + a * s2[..., 0] * c2[..., 1] * z
    grad = 2 * PI * a * c2[..., 0] * c2[..., 1] * z * PI * co[..., 0] * s[..., 1] * s[..., 2] \
        - 2 * PI * a * s2[..., 0] * s2[..., 1] * z * PI * s[..., 0] * co[..., 1] * s[..., 2] \
        + a * s2[..., 0] * c2[..., 1] * PI * s[..., 0] * s[..., 1] * co[..., 2]
    return 3 * PI ** 2 * k * u - grad + u


def _points(node, cell, bcs):
    return torch.einsum("qv,cvd->cqd", bcs, node[cell])


def _inputs(c, seed):
    """Mesh, space and the seed's coefficient data, before any form is built."""
    g = _generator(seed)
    mesh = _mesh(c, g)
    s = {"case": c, "mesh": mesh, "space": fa.LagrangeFESpace(mesh, c["p"])}
    s["a"], s["modes"] = _amplitudes(seed)
    nc = mesh.number_of_cells()
    if c["op"] == "elasticity":
        r = np.random.default_rng(seed)
        s["lam"], s["mu"] = float(r.uniform(0.5, 2.0)), float(r.uniform(0.3, 1.0))
    elif c["coef"] in ("cell", "cellexpr"):
        s["k"] = _lognormal(nc, g)
    elif c["coef"] == "point":       # a field already sampled at the quadrature points
        bcs = mesh.quadrature_formula(_quadrature(c)).get_quadrature_points_and_weights()[0].cuda()
        pts = _points(mesh.node, mesh.cell.long(), bcs)
        at = _source_at(pts, s["a"], s["modes"]) if c["op"] == "vector" else _diffusion_at(pts, s["a"])
        s["k"] = at.contiguous()
    if c["op"] == "spmv":
        n = s["space"].number_of_global_dofs()
        s["x"] = torch.randn(n, generator=g, device="cuda", dtype=torch.float64).to(DTYPES[c["dtype"]])
    return s


def _bilinear(s):
    c = s["case"]
    if c["op"] == "elasticity":
        return fa.BilinearForm(s["space"]).add_integrator(fa.LinearElasticityIntegrator(s["material"], q=c["q"] or None))
    k = _diffusion_expr(c["dim"], s["a"]) if c["coef"] == "expr" else s["k"]
    ints = [fa.ScalarDiffusionIntegrator(k, q=c["q"] or None)]
    if c["mass"]:
        ints.append(fa.ScalarMassIntegrator(1.0, q=c["q"] or None))
    return fa.BilinearForm(s["space"]).add_integrator(*ints)


def _linear(s, coef):
    c = s["case"]
    if coef == "expr":
        f = _source_expr(c["dim"], s["a"], s["modes"])
    elif coef == "cellexpr":
        f = 3 * PI ** 2 * expr.cell(s["k"]) * _sines(c["dim"])
    else:
        f = s["k"]
    return fa.LinearForm(s["space"]).add_integrator(fa.ScalarSourceIntegrator(f, q=c["q"] or None))


def _solve_source(c):
    """The manufactured source in 3D, the Fourier modes of a service request in 2D."""
    return "cellexpr" if c["dim"] == 3 else "expr"


def prepare(case, seed):
    s = _inputs(case, seed)
    op = case["op"]
    if op == "elasticity":
        gd = case["dim"]
        s["space"] = fa.TensorFunctionSpace(s["space"], (-1, gd))
        s["material"] = fa.LinearElasticMaterial("block", lame_lambda=s["lam"], shear_modulus=s["mu"],
                                                 **({} if gd == 3 else {"hypo": "plane_strain"}))
    if op == "element":
        method = "mfma_" + case["dtype"]
        s["group"] = fa.GroupIntegrator(fa.ScalarDiffusionIntegrator(s["k"], q=case["q"], method=method),
                                        fa.ScalarMassIntegrator(1.0, q=case["q"], method=method))
        return s
    pattern_of(s["space"])                       # the plan of every assembly on this space
    if op == "spmv":
        s["A"] = _bilinear(s).assembly(dtype=DTYPES[case["dtype"]])
    elif op == "dirichlet":
        s["A"] = _bilinear(s).assembly()
        s["F"] = _linear(s, "cellexpr").assembly()
        s["bc"] = fa.DirichletBC(s["space"], gd=_sines(case["dim"]) + 1.0)
    elif op == "solve":
        s["bc"] = fa.DirichletBC(s["space"], gd=_sines(case["dim"]))
        s["mg"] = GeometricMG(s["space"], s["bc"].is_boundary_dof, dtype=torch.float32)
    return s


def _csr(A):
    return [A.crow, A.col, A.values]


def run(s):
    c = s["case"]
    op = c["op"]
    if op == "matrix":
        return _csr(_bilinear(s).assembly(dtype=DTYPES[c["dtype"]]))
    if op == "vector":
        return _linear(s, c["coef"]).assembly()
    if op == "elasticity":
        return _csr(_bilinear(s).assembly())
    if op == "element":
        return s["group"].assembly(s["space"], dtype=torch.float32)
    if op == "dirichlet":
        A, F = s["bc"].apply(s["A"], s["F"])
        return _csr(A) + [F]
    if op == "spmv":
        return s["A"] @ s["x"]
    A = _bilinear(s).assembly()
    F = _linear(s, _solve_source(c)).assembly()
    if c["form"] == "refine":
        A2 = s["bc"].apply_matrix(A, dtype=torch.float32)
        s["mg"].setup(A2)
        return cg_refine(A, F, A2, s["mg"], s["bc"], rtol=1e-8, inner_rtol=1e-4)
    A2, F2 = s["bc"].apply(A, F)
    s["mg"].setup(A2)
    return fa.cg(A2, F2, M=s["mg"], atol=0.0, rtol=1e-8)


# ---- work and tolerance ---------------------------------------------------------
def _dofs(c):
    """Scalar DOFs: those of the grid refined p times, for either cell type."""
    n = 1
    for m in (c["nx"], c["ny"], c["nz"])[:c["dim"]]:
        n *= c["p"] * m + 1
    return n


#: mean stored entries of a row of a large grid's degree-p matrix
_ROW = {(2, 1): 7.0, (2, 2): 11.5, (2, 3): 16.3, (2, 4): 22.9, (3, 1): 14.8, (3, 2): 28.4, (3, 3): 46.0, (3, 4): 72.0}


def _nodes(c):
    n = 1
    for m in (c["nx"], c["ny"], c["nz"])[:c["dim"]]:
        n *= m + 1
    return n


def work(case):
    """Inputs read once and outputs written once: node coordinates (and, on a free mesh, the cell-to-DOF map), the
    coefficient, the row pointer and column indices that name the entries, the values or vector that come out."""
    c, dim, nc, n = case, case["dim"], _cells(case), _dofs(case)
    ld, nq = _ldof(c), math.comb(_quadrature(c) + dim - 1, dim)
    vb = 4 if c["dtype"] in ("f32", "fp32", "bf16") else 8
    nnz = _ROW[dim, c["p"]] * n
    geo = 8 * dim * _nodes(c) + (4 * nc * ld if c["mesh"] == "free" or c["p"] > 1 else 0)
    field = {"cell": 8 * nc, "cellexpr": 8 * nc, "point": 8 * nc * nq, "expr": 0}[c["coef"]]
    op = c["op"]
    if op == "matrix":
        return {"bytes": geo + field + 4 * n + vb * nnz, "flops": 2.0 * nc * ld * ld * (dim * (dim + 1) / 2 + 1)}
    if op == "vector":
        return {"bytes": geo + field + 8 * n, "flops": 2.0 * nc * nq * ld}
    if op == "elasticity":
        return {"bytes": geo + 4 * dim * n + 8 * dim * dim * nnz, "flops": 2.0 * nc * ld * ld * dim * dim * (dim + 1)}
    if op == "element":
        return {"bytes": geo + field + 4 * nc * ld * ld, "flops": 2.0 * nc * nq * 7 * ld * ld}
    if op == "dirichlet":
        return {"bytes": 12 * nnz + 8 * nnz + 24 * n, "flops": 2.0 * nnz}
    if op == "spmv":
        return {"bytes": (vb + 4) * nnz + (4 + 2 * vb) * n, "flops": 2.0 * nnz}
    # the matrix and right-hand side formed once, and ten iterations that read the FP32 operator once each
    return {"bytes": geo + 8 * nc + 12 * nnz + 10 * (8 * nnz + 16 * n), "flops": 10 * 4.0 * nnz}


def tolerance(case):
    op = case["op"]
    if op == "solve":
        return {"rel": 2e-8}                # both stop at 1e-8 of the right-hand side
    if op == "element":                     # BF16 inputs: 1.5e-3 from FP64 at P3 and P4
        return {"rel": 6e-3, "max": 5e-2} if case["dtype"] == "bf16" else {"rel": 5e-6}
    if case["dtype"] == "f32":
        return {"rel": 1e-6}
    return {"rel": 4e-15}                   # sums in another order (exact()) differ by 2e-16 to 4e-16


# ---- the same results in plain torch, FP64 -----------------------------------------
def _shape(bcs, p):
    """phi (NQ, ldof) and d phi / d lambda (NQ, ldof, dim + 1) of the Lagrange basis of degree p, local functions in
    the order of descending multi-indices."""
    d1 = bcs.shape[1]

    def indices(left, slots):
        return [(left,)] if slots == 1 else [(k,) + r for k in range(left, -1, -1) for r in indices(left - k, slots - 1)]

    lam = bcs.detach().clone().requires_grad_(True)
    phis, grads = [], []
    for alpha in indices(p, d1):
        f = torch.ones_like(lam[:, 0])
        for m, k in enumerate(alpha):
            for t in range(k):
                f = f * (p * lam[:, m] - t) / (t + 1)
        grads.append(torch.autograd.grad(f.sum(), lam)[0])
        phis.append(f.detach())
    return torch.stack(phis, 1), torch.stack(grads, 1)


def _geometry(node, cell):
    """(|T|, grad lambda (NC, dim + 1, dim))."""
    v = node[cell]
    J = v[:, 1:] - v[:, :1]                                    # rows: edges from vertex 0
    inv = torch.linalg.inv(J)                                  # columns: gradients of lambda_1..
    g = inv.transpose(1, 2)
    vol = torch.linalg.det(J) / math.factorial(J.shape[1])
    return vol, torch.cat([-g.sum(dim=1, keepdim=True), g], dim=1)


def _to_csr(c2d, elem, n):
    """(rows, cols, values) of the summed matrix, ordered by (row, column)."""
    key = (c2d.long()[:, :, None] * n + c2d.long()[:, None, :]).reshape(-1)
    uniq, inv = torch.unique(key, return_inverse=True)
    del key
    vals = torch.zeros(uniq.shape[0], dtype=torch.float64, device="cuda").index_add_(0, inv, elem.reshape(-1))
    return uniq // n, uniq % n, vals


def _rule(s):
    b, w = s["mesh"].quadrature_formula(_quadrature(s["case"])).get_quadrature_points_and_weights()
    return b.cuda(), w.cuda()


def _matrix_elements(s, take):
    c, node, cell = s["case"], s["mesh"].node, s["mesh"].cell.long()[take]
    bcs, w = _rule(s)
    phi, dphi = (t.cuda() for t in _shape(bcs, c["p"]))
    vol, gl = _geometry(node, cell)
    if c["coef"] == "expr":
        k = _diffusion_at(_points(node, cell, bcs), s["a"])
    else:
        k = s["k"][take] if s["k"].ndim == 2 else s["k"][take][:, None].expand(-1, w.shape[0])
    G = torch.einsum("qla,cad->cqdl", dphi, gl)
    nc, nq, dim, ld = G.shape
    G = G.reshape(nc, nq * dim, ld)
    kw = (k * w * vol[:, None])[:, :, None].expand(-1, -1, dim).reshape(nc, nq * dim, 1)
    K = torch.matmul(G.transpose(1, 2).contiguous(), G * kw)
    if c["mass"]:
        K = K + vol[:, None, None] * torch.einsum("q,qi,qj->ij", w, phi, phi)
    return K


def _chunked(s, f, size=100_000):
    nc = s["mesh"].number_of_cells()
    return torch.cat([f(s, slice(k, min(k + size, nc))) for k in range(0, nc, size)])


def _vector(s, coef):
    c, node, cell = s["case"], s["mesh"].node, s["mesh"].cell.long()
    bcs, w = _rule(s)
    phi = _shape(bcs, c["p"])[0]
    c2d = s["space"].cell_to_dof().long()
    out = torch.zeros(s["space"].number_of_global_dofs(), dtype=torch.float64, device="cuda")
    size = 200_000
    for b in range(0, cell.shape[0], size):
        t = slice(b, b + size)
        pts = _points(node, cell[t], bcs)
        if coef == "expr":
            f = _source_at(pts, s["a"], s["modes"])
        elif coef == "cellexpr":
            f = 3 * PI ** 2 * s["k"][t][:, None] * torch.sin(PI * pts).prod(dim=-1)
        else:
            f = s["k"][t] if s["k"].ndim == 2 else s["k"][t][:, None].expand(-1, w.shape[0])
        vol = _geometry(node, cell[t])[0]
        out.index_add_(0, c2d[t].reshape(-1), torch.matmul(f * w * vol[:, None], phi).reshape(-1))
    return out


def _dof_points(s):
    """Interpolation points of the space's DOFs."""
    c, node, cell = s["case"], s["mesh"].node, s["mesh"].cell.long()
    d1, p = cell.shape[1], c["p"]

    def indices(left, slots):
        return [(left,)] if slots == 1 else [(k,) + r for k in range(left, -1, -1) for r in indices(left - k, slots - 1)]

    bcs = torch.tensor(indices(p, d1), dtype=torch.float64, device="cuda") / p
    pts = torch.zeros((s["space"].number_of_global_dofs(), d1 - 1), dtype=torch.float64, device="cuda")
    c2d = s["space"].cell_to_dof().long()
    for i in range(bcs.shape[0]):
        pts[c2d[:, i]] = torch.einsum("v,cvd->cd", bcs[i], node[cell])
    return pts


def _fixed(pts):
    return ((pts < 1e-12) | (pts > 1 - 1e-12)).any(dim=1)


def _elasticity(s):
    c, node, cell = s["case"], s["mesh"].node, s["mesh"].cell.long()
    dim = c["dim"]
    bcs, w = _rule(s)
    dphi = _shape(bcs, c["p"])[1]
    M = torch.einsum("q,qia,qjb->ijab", w, dphi, dphi)
    out = []
    for b in range(0, cell.shape[0], 50_000):
        vol, gl = _geometry(node, cell[b:b + 50_000])
        S = torch.einsum("ijab,cad,cbe->cijde", M, gl, gl) * vol[:, None, None, None, None]   # d_d phi_i d_e phi_j
        tr = torch.diagonal(S, dim1=3, dim2=4).sum(-1)
        eye = torch.eye(dim, dtype=torch.float64, device="cuda")
        K = s["lam"] * S + s["mu"] * S.transpose(3, 4) + s["mu"] * tr[..., None, None] * eye
        out.append(K.permute(0, 1, 3, 2, 4).reshape(K.shape[0], dim * K.shape[1], -1))
    c2d = s["space"].cell_to_dof().long()
    c2d = (dim * c2d[:, :, None] + torch.arange(dim, device="cuda")).reshape(c2d.shape[0], -1)
    return _to_csr(c2d, torch.cat(out), dim * s["space"].number_of_global_dofs())


def _assembled(s):
    n = s["space"].number_of_global_dofs()
    return _to_csr(s["space"].cell_to_dof(), _chunked(s, _matrix_elements), n)


def _solution(s):
    """Jacobi-preconditioned CG on the assembled system, to the limit of FP64."""
    rows, cols, vals = _assembled(s)
    F = _vector(s, _solve_source(s["case"]))
    pts = _dof_points(s)
    fixed = _fixed(pts)
    g = torch.where(fixed, torch.sin(PI * pts).prod(dim=-1), torch.zeros_like(F))
    n = F.shape[0]
    count = torch.bincount(rows, minlength=n)
    start = torch.cumsum(count, 0) - count
    width = int(count.max())
    at = torch.arange(rows.shape[0], device="cuda") - start[rows]
    ecol = torch.zeros((n, width), dtype=torch.int64, device="cuda")
    eval_ = torch.zeros((n, width), dtype=torch.float64, device="cuda")
    ecol[rows, at], eval_[rows, at] = cols, vals
    diag = torch.zeros(n, dtype=torch.float64, device="cuda")
    diag[rows[rows == cols]] = vals[rows == cols]
    free = (~fixed).to(torch.float64)
    A = lambda v: (eval_ * v[ecol]).sum(dim=1) * free           # noqa: E731
    b = (F - (eval_ * g[ecol]).sum(dim=1)) * free
    x, r = torch.zeros_like(b), b.clone()
    z = r / diag
    p, rz = z.clone(), torch.dot(r, z)
    stop = 1e-14 * float(torch.linalg.norm(b))
    for k in range(20_000):
        Ap = A(p)
        alpha = rz / torch.dot(p, Ap)
        x += alpha * p
        r -= alpha * Ap
        z = r / diag
        rz_new = torch.dot(r, z)
        p = z + (rz_new / rz) * p
        rz = rz_new
        if k % 50 == 49 and float(torch.linalg.norm(r)) < stop:
            break
    return x + g


def exact(case, seed):
    s = _inputs(case, seed)
    op = case["op"]
    if op == "matrix":
        return [None, None, _assembled(s)[2]]
    if op == "vector":
        return _vector(s, case["coef"])
    if op == "elasticity":
        return [None, None, _elasticity(s)[2]]
    if op == "element":
        return _chunked(s, _matrix_elements)
    if op == "solve":
        return _solution(s)
    rows, cols, vals = _assembled(s)
    if op == "spmv":
        vals = vals.to(DTYPES[case["dtype"]]).double()           # the matrix in hand is the rounded one
        out = torch.zeros(s["space"].number_of_global_dofs(), dtype=torch.float64, device="cuda")
        return out.index_add_(0, rows, vals * s["x"].double()[cols])
    F = _vector(s, "cellexpr")
    pts = _dof_points(s)
    fixed = _fixed(pts)
    g = torch.where(fixed, torch.sin(PI * pts).prod(dim=-1) + 1.0, torch.zeros_like(F))
    out = F.index_add(0, rows, -vals * g[cols])
    keep = ~fixed[rows] & ~fixed[cols] | fixed[rows] & (rows == cols)
    vals = torch.where(fixed[rows], torch.ones_like(vals), vals)[keep]
    return [None, None, vals, torch.where(fixed, g, out)]
