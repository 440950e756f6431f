"""Rows summed from a record per cell (fa_assemble_p1_rows,
fa_assemble_elasticity_rows) against the element matrices of the same forms,
summed in FP64 on the CPU: meshes with shuffled numbering, a vertex of high
degree, the smallest meshes, both value types and DOF layouts.  An entry adds at
most `deg` cells' values, each a sum of at most 9 products on either side:
9 deg units in the last place of the largest entry."""
import threading

import numpy as np
import pytest
import torch

import fealpy_amd as fa
from fealpy_amd.fem import integrators, rows
from fealpy_amd.fem.pattern import pattern_of

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _shuffled(mesh, seed):
    g = np.random.default_rng(seed)
    node, cell = mesh.node.cpu().numpy(), mesh.cell.cpu().numpy()
    perm = g.permutation(len(node))
    new = np.empty_like(perm)
    new[perm] = np.arange(len(node))
    return type(mesh)(torch.as_tensor(node[perm], device=DEV), torch.as_tensor(new[cell][g.permutation(len(cell))],
                                                                              dtype=torch.int32, device=DEV))


def _fan(n):
    """n triangles around one vertex: a row of n + 1 entries and n incidences."""
    t = 2 * np.pi * np.arange(n) / n
    node = np.concatenate([[[0.0, 0.0]], np.stack([np.cos(t), np.sin(t)], 1)])
    cell = np.stack([np.zeros(n, int), 1 + np.arange(n), 1 + (np.arange(n) + 1) % n], 1)
    return fa.TriangleMesh(torch.as_tensor(node, device=DEV), torch.as_tensor(cell, dtype=torch.int32, device=DEV))


MESHES = {"tri1": lambda: fa.TriangleMesh.from_box(nx=1, ny=1, device=DEV),
          "tri": lambda: _shuffled(fa.TriangleMesh.from_box(nx=9, ny=7, device=DEV), 1),
          "fan": lambda: _fan(300),
         "fan100": lambda: _fan(100),
          "tet1": lambda: _shuffled(fa.TetrahedronMesh.from_box(nx=1, ny=1, nz=1, device=DEV), 2),
          "tet2": lambda: _shuffled(fa.TetrahedronMesh.from_box(nx=2, ny=1, nz=2, device=DEV), 5),
         "tet": lambda: _shuffled(fa.TetrahedronMesh.from_box(nx=4, ny=3, nz=5, device=DEV), 3)}


def _dense(space, elem):
    n = space.number_of_global_dofs()
    c2d = space.cell_to_dof().cpu().long()
    out = torch.zeros(n * n, dtype=torch.float64)
    out.index_add_(0, (c2d[:, :, None] * n + c2d[:, None, :]).reshape(-1), elem.cpu().reshape(-1))
    return out.reshape(n, n), int(torch.bincount(c2d.reshape(-1)).max())


def _check(A, space, elem, dtype):
    ref, deg = _dense(space, elem)
    eps = 9 * deg * 2.2e-16 + (6e-8 if dtype == torch.float32 else 0.0)
    assert A.values.dtype == dtype
    assert float((A.to_dense().cpu().double() - ref).abs().max()) <= eps * float(ref.abs().max())


@pytest.mark.parametrize("name", sorted(MESHES))
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("ops", ["diff", "mass", "both"])
def test_p1_rows(name, dtype, ops, monkeypatch):
    monkeypatch.setattr(integrators, "RECORDS_MIN_CELLS", 0)
    mesh, calls = MESHES[name](), []
    monkeypatch.setattr(integrators, "p1_values", lambda *a: calls.append(rows.p1_values(*a)) or calls[-1])
    space = fa.LagrangeFESpace(mesh, 1)
    k = torch.as_tensor(np.exp(np.random.default_rng(4).standard_normal(mesh.number_of_cells())), device=DEV)
    ints = [fa.ScalarDiffusionIntegrator(k, q=3)] if ops != "mass" else []
    ints += [fa.ScalarMassIntegrator(0.5 if ops == "both" else k, q=3)] if ops != "diff" else []
    group = fa.GroupIntegrator(*ints)
    A = fa.BilinearForm(space).add_integrator(group).assembly(dtype=dtype)
    # rows of more than 128 entries are summed from element matrices
    assert [v is not None for v in calls] == ([] if name == "fan" else [True])
    _check(A, space, group.assembly(space), dtype)


@pytest.mark.parametrize("name,p", [("tri1", 1), ("tri", 1), ("tri", 2), ("fan", 2), ("tri", 3), ("tri", 4), ("tet1", 1),
                                    ("tet", 1), ("tet1", 2), ("tet", 2), ("tet", 3)])
@pytest.mark.parametrize("prio", [False, True])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_elasticity_rows(name, p, prio, dtype, monkeypatch):
    monkeypatch.setattr(rows, "ELASTICITY_MIN_DOFS", 0)
    mesh = MESHES[name]()
    gd = mesh.geo_dimension()
    space = fa.TensorFunctionSpace(fa.LagrangeFESpace(mesh, p), (gd, -1) if prio else (-1, gd))
    mat = fa.LinearElasticMaterial("m", lame_lambda=1.3, shear_modulus=0.7,
                                   **({} if gd == 3 else {"hypo": "plane_strain"}))
    it = fa.LinearElasticityIntegrator(mat, q=p + 2)
    assert rows.elasticity_values(space, it, dtype) is not None
    A = fa.BilinearForm(space).add_integrator(it).assembly(dtype=dtype)
    _check(A, space, it.assembly(space), dtype)


@pytest.mark.parametrize("vector", [False, True])
def test_first_assembly_from_two_streams(vector, monkeypatch):
    """Two threads, a stream each, assemble on a space whose tables and row positions neither has built yet."""
    monkeypatch.setattr(integrators, "RECORDS_MIN_CELLS", 0)
    monkeypatch.setattr(rows, "ELASTICITY_MIN_DOFS", 0)
    mesh = MESHES["tet"]()
    mat = fa.LinearElasticMaterial("m", lame_lambda=1.3, shear_modulus=0.7)

    def assembled(space):
        if vector:
            space = fa.TensorFunctionSpace(space, (-1, 3))
            return fa.BilinearForm(space).add_integrator(fa.LinearElasticityIntegrator(mat, q=4)).assembly().values
        return fa.BilinearForm(space).add_integrator(fa.ScalarDiffusionIntegrator(2.0, q=3)).assembly().values

    ref = assembled(fa.LagrangeFESpace(mesh, 2 if vector else 1))
    for _ in range(4):
        rows._elasticity_tables.cache_clear()
        space, out, start = fa.LagrangeFESpace(mesh, 2 if vector else 1), [None, None], threading.Barrier(2)
        torch.cuda.synchronize()

        def work(i):
            with torch.cuda.stream(torch.cuda.Stream()):
                start.wait()
                out[i] = assembled(space)
                torch.cuda.current_stream().synchronize()

        threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert torch.equal(out[0], ref) and torch.equal(out[1], ref)


@pytest.mark.parametrize("p,n", [(1, 980), (1, 2700), (2, 700), (2, 1300)])
def test_long_rows_sum_from_elements(p, n):
    """One vertex of very many triangles: rows longer than 64 / ldof of them would fit in LDS."""
    fan = _fan(n)
    cell = (fan.cell + n) % (n + 1)          # the centre last: the edge builder takes 1024 edges from their smallest vertex
    space = fa.LagrangeFESpace(fa.TriangleMesh(fan.node.roll(-1, 0).contiguous(), cell.to(torch.int32)), p)
    it = fa.ScalarDiffusionIntegrator(2.0, q=p + 1)
    for dtype in (torch.float64, torch.float32):
        for _ in range(2):
            _check(fa.BilinearForm(space).add_integrator(it).assembly(dtype=dtype), space, it.assembly(space), dtype)


@pytest.mark.parametrize("name,p,vector", [("tri", 3, False), ("tet", 2, False), ("tri", 4, True), ("tet2", 3, True),
                                           ("tet1", 4, True), ("tet2", 4, True)])
def test_rows_sum_in_cell_order(name, p, vector, monkeypatch):
    """Every entry adds its cells' values one after another in ascending cell order, also where an element row is
    wider than a wave (105 columns): bit for bit np.add.at."""
    mesh = MESHES[name]()
    gd = mesh.geo_dimension()
    space = fa.LagrangeFESpace(mesh, p)
    it = fa.ScalarDiffusionIntegrator(2.0, q=p + 1)
    if vector:
        space = fa.TensorFunctionSpace(space, (-1, gd))
        it = fa.LinearElasticityIntegrator(fa.LinearElasticMaterial("m", lame_lambda=1.3, shear_modulus=0.7,
                                                                    **({} if gd == 3 else {"hypo": "plane_strain"})))
        monkeypatch.setattr(rows, "elasticity_values", lambda *a: None)
    n, c2d = space.number_of_global_dofs(), space.cell_to_dof().cpu().numpy()
    ref = np.zeros((n, n))
    np.add.at(ref, (c2d[:, :, None], c2d[:, None, :]), it.assembly(space).cpu().numpy())
    for _ in range(2):           # the columns searched, then their kept positions
        assert np.array_equal(fa.BilinearForm(space).add_integrator(it).assembly().to_dense().cpu().numpy(), ref)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_positions_from_the_second_sum(dtype):
    """A space assembled once keeps no row positions and waits for nothing; the next sums have the same bits.  While a
    stream captures nothing is built either."""
    mesh = MESHES["tet"]()
    it = fa.ScalarDiffusionIntegrator(2.0, q=3)
    space = fa.LagrangeFESpace(mesh, 2)
    first = fa.BilinearForm(space).add_integrator(it).assembly(dtype=dtype).values
    assert pattern_of(space)._pos is None
    graph, out = torch.cuda.CUDAGraph(), None
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = fa.BilinearForm(space).add_integrator(it).assembly(dtype=dtype).values
    assert pattern_of(space)._pos is None
    second = fa.BilinearForm(space).add_integrator(it).assembly(dtype=dtype).values
    assert pattern_of(space)._pos is not None
    assert torch.equal(first, second)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, first)
