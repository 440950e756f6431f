"""FP64 element matrices on the matrix instruction (fa_element_matrices) and
their sum into CSR rows (fa_sum_rows): cell counts around a block's groups,
rules larger than its staged points, every kind of coefficient.  The oracle is
the plain FP64 sum in torch on the CPU; both add NQ TD (TD + 1) / 2 products, so
they differ by that many units in the last place of the largest entry at most."""
import math

import numpy as np
import pytest
import torch

import fealpy_amd as fa
from fealpy_amd import expr
from fealpy_amd.fem import integrators
from fealpy_amd.functionspace.basis import grad_shape_function, shape_function

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _mesh(dims):
    if len(dims) == 2:
        return fa.TriangleMesh.from_box(nx=dims[0], ny=dims[1], device=DEV)
    return fa.TetrahedronMesh.from_box(nx=dims[0], ny=dims[1], nz=dims[2], device=DEV)


def _coefficient(kind, nc, nq, gen):
    """(what the integrator takes, values (NC, NQ) of a function of the points)"""
    if kind == "none":
        return None, lambda pts: torch.ones(nc, nq, dtype=torch.float64)
    if kind == "cell":
        k = torch.rand(nc, generator=gen, dtype=torch.float64) + 0.5
        return k.to(DEV), lambda pts: k[:, None].expand(-1, nq)
    if kind == "point":
        k = torch.rand((nc, nq), generator=gen, dtype=torch.float64) + 0.5
        return k.to(DEV), lambda pts: k
    f = 1.0 + 0.5 * expr.sin(math.pi * expr.x) * expr.cos(2.0 * expr.y)
    return f, lambda pts: f(pts)


def _reference(mesh, p, q, kd, km):
    bcs, w = (t.cpu() for t in mesh.quadrature_formula(q).get_quadrature_points_and_weights())
    v = mesh.node.cpu()[mesh.cell.cpu().long()]
    J = v[:, 1:] - v[:, :1]
    vol = torch.linalg.det(J) / math.factorial(J.shape[1])
    g = torch.linalg.inv(J).transpose(1, 2)
    gl = torch.cat([-g.sum(1, keepdim=True), g], dim=1)
    pts = torch.einsum("qv,cvd->cqd", bcs, v)
    out = 0.0
    if kd is not None:
        G = torch.einsum("qla,cad->cqld", torch.as_tensor(grad_shape_function(bcs.numpy(), p)), gl)
        out = torch.einsum("q,cq,c,cqid,cqjd->cij", w, kd(pts), vol, G, G)
    if km is not None:
        phi = torch.as_tensor(shape_function(bcs.numpy(), p))
        out = out + torch.einsum("q,cq,c,qi,qj->cij", w, km(pts), vol, phi, phi)
    return out


SHAPES = [((1, 1), 1, 4), ((4, 8), 2, 5), ((3, 11), 3, 6), ((5, 7), 4, 9), ((2, 3), 2, 11), ((1, 1, 1), 1, 4),
          ((2, 2, 3), 2, 5), ((3, 1, 4), 3, 5), ((2, 1, 3), 4, 6), ((1, 2, 3), 4, 7), ((1, 2, 1), 3, 9), ((2, 1, 1), 1, 9)]


@pytest.mark.parametrize("dims,p,q", SHAPES)
@pytest.mark.parametrize("diff,mass", [("cell", None), (None, "cell"), ("point", None), (None, "point"), ("sep", "none"),
                                       ("cell", "sep"), ("point", "cell"), ("none", "point"), ("sep", "point")])
def test_element_and_assembled_matrices(dims, p, q, diff, mass):
    mesh = _mesh(dims)
    space = fa.LagrangeFESpace(mesh, p)
    nc = mesh.number_of_cells()
    nq = mesh.quadrature_formula(q).get_quadrature_points_and_weights()[1].shape[0]
    gen = torch.Generator().manual_seed(5)
    ints, ref = [], {"diff": None, "mass": None}
    for name, kind, cls in (("diff", diff, fa.ScalarDiffusionIntegrator), ("mass", mass, fa.ScalarMassIntegrator)):
        if kind is not None:
            coef, ref[name] = _coefficient(kind, nc, nq, gen)
            ints.append(cls(coef, q=q))
    group = fa.GroupIntegrator(*ints)
    K = _reference(mesh, p, q, ref["diff"], ref["mass"])
    bound = nq * len(dims) * (len(dims) + 1) / 2 * 2.2e-16 * float(K.abs().max())
    got = group.assembly(space).cpu()
    assert float((got - K).abs().max()) <= bound
    assert float((group.assembly(space, dtype=torch.float32).cpu().double() - K).abs().max()) \
        <= bound + 6e-8 * float(K.abs().max())
    n = space.number_of_global_dofs()
    c2d = space.cell_to_dof().cpu().long()
    full = torch.zeros(n * n, dtype=torch.float64)
    full.index_add_(0, (c2d[:, :, None] * n + c2d[:, None, :]).reshape(-1), K.reshape(-1))
    for _ in range(2):           # the columns searched, then their kept positions (fa_sum_rows)
        A = fa.BilinearForm(space).add_integrator(*ints).assembly()
        assert float((A.to_dense().cpu().reshape(-1) - full).abs().max()) <= 24 * bound   # at most 24 cells an entry


def test_region_sums_like_the_whole():
    """A region's pattern is summed by the searching kernel: the two halves add up to the matrix of all cells."""
    mesh = _mesh((3, 2, 3))
    space = fa.LagrangeFESpace(mesh, 2)
    nc = mesh.number_of_cells()
    half = torch.arange(nc, device=DEV) < nc // 2
    parts = [fa.BilinearForm(space).add_integrator(fa.ScalarDiffusionIntegrator(2.0, q=4, region=r)).assembly().to_dense()
             for r in (half, ~half)]
    A = fa.BilinearForm(space).add_integrator(fa.ScalarDiffusionIntegrator(2.0, q=4)).assembly().to_dense()
    assert float((parts[0] + parts[1] - A).abs().max()) <= 24 * 2.2e-16 * float(A.abs().max())


@pytest.mark.parametrize("td,p,q", [(2, 2, 5), (2, 3, 6), (2, 4, 7), (3, 1, 4), (3, 2, 5), (3, 3, 6), (3, 4, 7)])
@pytest.mark.parametrize("op", ["diff", "mass"])
def test_reference_sums_keep_their_precision(td, p, q, op):
    """The reference simplex, whose gradients are exact, against sums with 64 bits of mantissa: four roundings an entry
    (the table's, |T|'s, their product, the sum of the pairs) of 2^-53 at most, 1.2 of it in the mean square; 2 allowed.
    Sums over the points in plain order were 2.3 to 6.5 off (every cell repeats them)."""
    node = torch.cat([torch.zeros(1, td), torch.eye(td)]).double().to(DEV)
    cell = torch.arange(td + 1, dtype=torch.int32, device=DEV)[None]
    mesh = (fa.TriangleMesh if td == 2 else fa.TetrahedronMesh)(node, cell)
    bcs, w = (t.cpu().numpy() for t in mesh.quadrature_formula(q).get_quadrature_points_and_weights())
    R = grad_shape_function(bcs, p).astype(np.longdouble)
    R = R[:, :, 1:] - R[:, :, :1] if op == "diff" else shape_function(bcs, p).astype(np.longdouble)[:, :, None]
    ref = np.einsum("q,qia,qja->ij", w.astype(np.longdouble), R, R) / math.factorial(td)
    cls = fa.ScalarDiffusionIntegrator if op == "diff" else fa.ScalarMassIntegrator
    got = cls(torch.ones(1, dtype=torch.float64, device=DEV), q=q).assembly(fa.LagrangeFESpace(mesh, p))[0].cpu().numpy()
    assert np.sqrt(((got - ref) ** 2).sum() / (ref ** 2).sum()) <= 2 * 2.0 ** -53


@pytest.mark.parametrize("dims,p", [((5, 4), 2), ((2, 3, 2), 2), ((1, 2, 1), 3), ((3, 3), 4)])
def test_separable_coefficient_sampled_or_in_the_kernel(dims, p, monkeypatch):
    """Both routes evaluate the same factors in the same order: the same bits."""
    space = fa.LagrangeFESpace(_mesh(dims), p)
    f = 1.0 + 0.5 * expr.sin(math.pi * expr.x) * expr.cos(2.0 * expr.y) + expr.exp(expr.x) * expr.y
    it = fa.ScalarDiffusionIntegrator(f, q=p + 2)
    out = []
    for sampled in (True, False):
        monkeypatch.setattr(integrators, "_sampled_first", lambda points, ldof: sampled)
        out.append(it.assembly(space))
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("dims,p,q", [((15, 15, 15), 4, 7), ((30, 30, 30), 2, 11), ((260, 260), 2, 13)])
@pytest.mark.parametrize("diff,mass", [("point", "point"), ("point", "cell")])
def test_second_group_of_a_block(dims, p, q, diff, mass):
    """More cells than one round of the capped grid, with rules of several chunks: a block stages the first points'
    tables again for its next group.  The same cells alone, one group a block, have the same bits."""
    mesh = _mesh(dims)
    nc = mesh.number_of_cells()
    nq = mesh.quadrature_formula(q).get_quadrature_points_and_weights()[1].shape[0]
    assert nq > (56 if p == 4 else 64)
    gen = torch.Generator(device=DEV).manual_seed(7)
    kd = torch.rand((nc, nq), generator=gen, device=DEV, dtype=torch.float64) + 0.5
    km = torch.rand((nc, nq) if mass == "point" else nc, generator=gen, device=DEV, dtype=torch.float64) + 0.5
    idx = torch.arange(nc - 1, 0, -max(nc // 500, 1), device=DEV)

    def elements(a, b, indices):
        return fa.GroupIntegrator(fa.ScalarDiffusionIntegrator(a, q=q), fa.ScalarMassIntegrator(b, q=q)).assembly(
            fa.LagrangeFESpace(mesh, p), indices=indices)

    assert torch.equal(elements(kd, km, None)[idx], elements(kd[idx].contiguous(), km[idx].contiguous(), idx))
