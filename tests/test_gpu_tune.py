"""The project autotuner (fealpy_amd.tune): it picks one of the candidate
tiles by measurement, stores it in the library's table and its cache file,
and the choice never changes assembled values (pass 2 sums in incidence
order for every lane count); the CSR SpMV agrees across choices to rounding."""
import json

import numpy as np
import pytest
import torch

import fealpy_amd as fa
from fealpy_amd import _native as nat
from fealpy_amd.tune import CANDIDATES, SPMV_LANES, SUM_ROWS_LANES, Autotuner

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def test_assembly_lanes_bitwise_and_cached(tmp_path, monkeypatch):
    from fealpy_amd.fem import integrators
    monkeypatch.setattr(integrators, "BOX_ASSEMBLY", False)     # the two-pass kernels, not the from_box one
    L = nat.lib()
    mesh = fa.TetrahedronMesh.from_box(nx=24, ny=24, nz=20, device=DEV)     # 69,120 cells: two-pass path
    space = fa.LagrangeFESpace(mesh, 1)
    k = torch.as_tensor(np.exp(np.random.default_rng(9).standard_normal(mesh.number_of_cells())), device=DEV)
    from fealpy_amd.fem.pattern import pattern_of
    key = L.fa_tune_key(SUM_ROWS_LANES, 3, pattern_of(space).max_row)
    vals = {}
    try:
        for g in CANDIDATES[SUM_ROWS_LANES]:
            nat.check(L.fa_tune_set(SUM_ROWS_LANES, key, g), "fa_tune_set")
            vals[g] = fa.BilinearForm(space).add_integrator(fa.ScalarDiffusionIntegrator(k, q=2)).assembly().values
        ref = vals[8]
        for g, v in vals.items():
            assert torch.equal(v, ref), g
        path = tmp_path / "tune.json"
        t = Autotuner(path=str(path), reps=3)
        best, ms = t.tune_assembly(space, k, q=2)
        assert best in CANDIDATES[SUM_ROWS_LANES] and set(ms) == set(CANDIDATES[SUM_ROWS_LANES])
        assert L.fa_tune_get(SUM_ROWS_LANES, key) == best
        data = json.loads(path.read_text())
        dev = data[torch.cuda.get_device_name(DEV)]
        assert dev["sum_rows_lanes"][str(key)] == best
        nat.check(L.fa_tune_set(SUM_ROWS_LANES, key, 0), "fa_tune_set")
        assert Autotuner(path=str(path)).apply_cached(DEV) >= 1
        assert L.fa_tune_get(SUM_ROWS_LANES, key) == best
    finally:
        nat.check(L.fa_tune_set(SUM_ROWS_LANES, key, 0), "fa_tune_set")


def test_assembly_tuning_times_the_two_passes(monkeypatch):
    """Also on a mesh large enough to be assembled from a record per cell, where the lane count changes nothing."""
    from fealpy_amd.fem import integrators
    monkeypatch.setattr(integrators, "RECORDS_MIN_CELLS", 0)

    def refuse(*args):
        raise AssertionError("rows from records")
    monkeypatch.setattr(integrators, "p1_values", refuse)
    space = fa.LagrangeFESpace(fa.TetrahedronMesh.from_box(nx=5, ny=4, nz=3, device=DEV), 1)
    L = nat.lib()
    from fealpy_amd.fem.pattern import pattern_of
    key = L.fa_tune_key(SUM_ROWS_LANES, 3, pattern_of(space).max_row)
    try:
        Autotuner(path=None, reps=1).tune_assembly(space, q=2)
    finally:
        nat.check(L.fa_tune_set(SUM_ROWS_LANES, key, 0), "fa_tune_set")
    assert integrators.RECORDS_MIN_CELLS == 0 and integrators.BOX_ASSEMBLY


def test_spmv_lanes(tmp_path):
    L = nat.lib()
    mesh = fa.TetrahedronMesh.from_box(nx=12, ny=12, nz=12, device=DEV)
    space = fa.LagrangeFESpace(mesh, 2)
    A = fa.BilinearForm(space).add_integrator(fa.ScalarDiffusionIntegrator(q=3)).assembly()
    key = L.fa_tune_key(SPMV_LANES, A.shape[0], A.nnz)
    x = torch.rand(A.shape[0], dtype=torch.float64, device=DEV)
    try:
        ys = {}
        for g in CANDIDATES[SPMV_LANES]:
            nat.check(L.fa_tune_set(SPMV_LANES, key, g), "fa_tune_set")
            ys[g] = A @ x
        ref = ys[CANDIDATES[SPMV_LANES][0]]
        for g, y in ys.items():
            assert float((y - ref).abs().max()) <= 1e-13 * float(ref.abs().max()), g
        best, _ = Autotuner(path=str(tmp_path / "t.json"), reps=3).tune_spmv(A)
        assert best in CANDIDATES[SPMV_LANES] and L.fa_tune_get(SPMV_LANES, key) == best
    finally:
        nat.check(L.fa_tune_set(SPMV_LANES, key, 0), "fa_tune_set")


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("mean", [1, 3, 8, 9, 16, 17, 40, 130, 300])
def test_spmv_every_lane_count_is_a_candidate(mean, dtype):
    """The built-in choice is among the candidates, one class each, and every candidate gives the same product."""
    L, n = nat.lib(), 400
    key = L.fa_tune_key(SPMV_LANES, n, n * mean)
    default = next(g for g in (1, 2, 4, 8, 16, 32, 64) if g == 64 or mean <= 8 * g)
    assert default in CANDIDATES[SPMV_LANES] and key == (1, 2, 4, 8, 16, 32, 64).index(default)
    g = np.random.default_rng(mean)
    col = np.stack([np.sort(g.choice(n, mean, replace=False)) for _ in range(n)])
    val = g.standard_normal((n, mean))
    A = fa.CSRTensor(torch.arange(n + 1, dtype=torch.int32, device=DEV) * mean,
                     torch.as_tensor(col.reshape(-1), dtype=torch.int32, device=DEV),
                     torch.as_tensor(val.reshape(-1), dtype=dtype, device=DEV), (n, n))
    x = torch.as_tensor(g.standard_normal(n), dtype=dtype, device=DEV)
    v, xs = A.values.cpu().double().numpy().reshape(n, mean), x.cpu().double().numpy()
    ref, size = (v * xs[col]).sum(1), (np.abs(v * xs[col])).sum(1)
    eps = 2.2e-16 if dtype == torch.float64 else 6e-8
    try:
        for lanes in (0, *CANDIDATES[SPMV_LANES]):
            nat.check(L.fa_tune_set(SPMV_LANES, key, lanes), "fa_tune_set")
            # FP64: the reference adds `mean` terms; FP32: one rounding of the result
            assert np.all(np.abs((A @ x).cpu().double().numpy() - ref) <= eps * (mean if eps < 1e-9 else 1.01) * size)
    finally:
        nat.check(L.fa_tune_set(SPMV_LANES, key, 0), "fa_tune_set")


def test_tune_set_rejects_bad_family():
    L = nat.lib()
    assert L.fa_tune_set(7, 0, 8) == nat.FA_EINVAL
    assert L.fa_tune_key(7, 1, 1) == -1
