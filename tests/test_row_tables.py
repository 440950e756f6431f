"""Reference tables of the row kernels: p1_table formed on the host and complete
when it is published, each entry the exact sum of the rule's numbers to half a
unit in the last place (and a tenth, for sums of 64 mantissa bits); the
elasticity table the element kernel's, reduced, within (NQ + 4) units of that
table's largest entry."""
from fractions import Fraction

import numpy as np
import pytest
import torch

import fealpy_amd as fa
from fealpy_amd.fem import rows
from fealpy_amd.functionspace.basis import grad_shape_function, shape_function


def _space(td, p):
    mesh = fa.TriangleMesh.from_box(nx=1, ny=1) if td == 2 else fa.TetrahedronMesh.from_box(nx=1, ny=1, nz=1)
    return fa.LagrangeFESpace(mesh, p)


def _exact(space, q):
    """(M[a][b][i][j], mass[i][j]) as exact fractions of the rule's and basis' FP64 numbers."""
    b, w = (t.numpy() for t in space.mesh.quadrature_formula(q).get_quadrature_points_and_weights())
    F = np.vectorize(Fraction, otypes=[object])
    R, phi, w = F(grad_shape_function(b, space.p)), F(shape_function(b, space.p)), F(w)
    R = R[:, :, 1:] - R[:, :, :1]
    return np.einsum("q,qia,qjb->abij", w, R, R), np.einsum("q,qi,qj->ij", w, phi, phi)


@pytest.mark.parametrize("td,q", [(2, 2), (2, 4), (3, 2), (3, 4), (3, 6)])
def test_p1_table_is_exact_to_rounding(td, q):
    space = _space(td, 1)
    M, mass = _exact(space, q)
    pairs = [(a, b) for a in range(td) for b in range(a, td)]
    exact = np.stack([M[a, b] if a == b else M[a, b] + M[b, a] for a, b in pairs] + [mass])
    for g, e in zip(rows.p1_table(space, q).reshape(-1).tolist(), exact.reshape(-1)):
        assert abs(Fraction(g) - e) <= Fraction(1.1 * 2.0 ** -53 * max(abs(float(e)), 1e-3))


@pytest.mark.parametrize("td,p,q", [(2, 1, 4), (3, 1, 4), (2, 2, 5), (3, 2, 5), (2, 4, 7)])
def test_elasticity_table_reduces_the_element_kernels(td, p, q):
    space = _space(td, p)
    M, reduced = rows.elasticity_tables(space, q)
    nq = len(rows._rule(space, q)[1])
    exact = np.vectorize(float)(_exact(space, q)[0])
    assert float(np.abs(reduced.numpy() - exact).max()) <= (nq + 4) * 2.0 ** -52 * float(M.abs().max())


def test_p1_table_queues_no_device_work(monkeypatch):
    """A kernel of the building stream would leave the published table incomplete for any other stream."""
    def refuse(*args, **kw):
        raise AssertionError("a table formed by queued tensor operations")

    space = _space(3, 1)
    for name in ("einsum", "stack", "matmul"):
        monkeypatch.setattr(torch, name, refuse)
    rows.p1_table(space, 3)
