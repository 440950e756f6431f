"""Element vectors (fa_element_vectors) where the block's tiling can go wrong:
cell counts around its batch, rules larger than its staged points, and
separable sources whose factors repeat, fill or exceed the block's table.
The oracle is the plain FP64 sum of the same integrand in torch on the CPU;
both sides add NQ products of O(1) terms, so they differ by NQ units in the
last place at most: NQ * 2.2e-16 relative to the largest entry, plus 4e-15 of
the sines' own rounding."""
import math

import pytest
import torch

import fealpy_amd as fa
from fealpy_amd import expr
from fealpy_amd.functionspace.basis import shape_function

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")
NAN = float("nan")
PI = math.pi


def many_arguments(n):
    """n distinct sine arguments (one table column each) over two coordinates."""
    f = None
    for k in range(1, n // 2 + 1):
        t = (0.5 / k) * expr.sin(k * PI * expr.x) * expr.sin((k + 0.5) * expr.y)
        f = t if f is None else f + t
    return f


SOURCES = {
    "repeats": 2.0 * expr.sin(PI * expr.x) * expr.cos(PI * expr.x) * expr.cos(PI * expr.y) + expr.exp(-1.0 * expr.x)
    * expr.sin(2.0 * expr.y) * expr.cos(2.0 * expr.y) * expr.sin(PI * expr.x) * expr.y + expr.x * expr.x * expr.x + 0.5,
    "fills": many_arguments(16),
    "exceeds": many_arguments(20),
}


def _mesh(dim, dims):
    if dim == 2:
        return fa.TriangleMesh.from_box(nx=dims[0], ny=dims[1], device=DEV)
    return fa.TetrahedronMesh.from_box(nx=dims[0], ny=dims[1], nz=dims[2], device=DEV)


def _reference(mesh, p, q, values):
    """|T| sum_q w_q f(x_cq) phi_i(q) on the CPU; values(points (NC, NQ, GD))."""
    bcs, w = (t.cpu() for t in mesh.quadrature_formula(q).get_quadrature_points_and_weights())
    v = mesh.node.cpu()[mesh.cell.cpu().long()]
    vol = torch.linalg.det(v[:, 1:] - v[:, :1]) / math.factorial(v.shape[2])
    phi = torch.as_tensor(shape_function(bcs.numpy(), p))
    f = values(torch.einsum("qv,cvd->cqd", bcs, v))
    return vol[:, None] * torch.einsum("q,cq,qi->ci", w, f, phi)


@pytest.mark.parametrize("dim,dims,p,q", [(2, (1, 1), 1, 4), (2, (8, 4), 1, 4), (2, (5, 13), 2, 5), (2, (7, 9), 4, 11),
                                          (3, (1, 1, 1), 1, 2), (3, (2, 3, 4), 2, 5), (3, (3, 2, 6), 3, 6),
                                          (3, (2, 2, 3), 4, 7), (3, (1, 2, 1), 2, 9), (3, (1, 1, 2), 1, 11)])
@pytest.mark.parametrize("name", sorted(SOURCES))
def test_element_vectors_match_plain_sums(dim, dims, p, q, name):
    mesh = _mesh(dim, dims)
    space = fa.LagrangeFESpace(mesh, p)
    f = SOURCES[name]
    got = fa.ScalarSourceIntegrator(f, q=q).assembly(space).cpu()
    ref = _reference(mesh, p, q, lambda pts: f(pts))
    nq = mesh.quadrature_formula(q).get_quadrature_points_and_weights()[1].shape[0]
    assert float((got - ref).abs().max()) <= (nq * 2.2e-16 + 4e-15) * float(ref.abs().max())


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_sampled_source_and_its_sum(dtype):
    """A (NC, NQ) source, and the gathered vector against index_add."""
    mesh = _mesh(3, (3, 4, 2))
    space = fa.LagrangeFESpace(mesh, 3)
    nq = mesh.quadrature_formula(5).get_quadrature_points_and_weights()[1].shape[0]
    f = torch.rand((mesh.number_of_cells(), nq), generator=torch.Generator().manual_seed(3), dtype=torch.float64)
    ref = _reference(mesh, 3, 5, lambda pts: f)
    full = torch.zeros(space.number_of_global_dofs(), dtype=torch.float64)
    full.index_add_(0, space.cell_to_dof().cpu().long().reshape(-1), ref.reshape(-1))
    got = fa.LinearForm(space).add_integrator(fa.ScalarSourceIntegrator(f.to(DEV), q=5)).assembly(dtype=dtype).cpu()
    eps = 2.2e-16 if dtype == torch.float64 else 1.2e-7 / 35     # one rounding of each element value and add
    assert float((got.double() - full).abs().max()) <= 2 * 35 * eps * float(full.abs().max())


@pytest.mark.parametrize("factor", [lambda s, a, b: expr.sin(a * s + b), lambda s, a, b: expr.cos(a * s + b),
                                    lambda s, a, b: expr.exp(a * s + b), lambda s, a, b: a * s + b])
@pytest.mark.parametrize("a,b", [(NAN, 0.5), (2.0, NAN), (NAN, NAN)])
def test_nan_parameters(factor, a, b):
    """A factor with a NaN in it makes its term NaN at every point, beside terms of other factors, and reaches
    nothing else: the same forms without it are as they were."""
    mesh = fa.TriangleMesh.from_box(nx=9, ny=8, device=DEV)
    space = fa.LagrangeFESpace(mesh, 2)
    other = 1.0 + expr.exp(expr.x) * expr.sin(2.0 * expr.y) + expr.cos(expr.x) * (expr.y + 2.0)

    def forms(f):
        return (fa.LinearForm(space).add_integrator(fa.ScalarSourceIntegrator(f, q=4)).assembly(),
                fa.BilinearForm(space).add_integrator(fa.ScalarDiffusionIntegrator(f, q=4)).assembly().values)

    before = forms(other)
    for out in forms(other + factor(expr.x, a, b) * expr.cos(expr.y)):
        assert bool(torch.isnan(out).all())
    for out, ref in zip(forms(other), before):
        assert torch.equal(out, ref) and bool(torch.isfinite(out).all())
