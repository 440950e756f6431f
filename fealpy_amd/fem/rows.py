"""CSR rows straight from a record per cell (fa_assemble_p1_rows,
fa_assemble_elasticity_rows) on a space's own pattern: P1 diffusion and mass
with coefficients constant on each cell, and isotropic elasticity of any
degree.  No array of element matrices is formed (the reference's
``integrator.assembly`` -> COO -> coalesce, fem/bilinear_form.py:46-105)."""
import functools

import numpy as np
import torch

from .. import _native as nat
from ..functionspace.basis import grad_shape_function, shape_function
from .pattern import pattern_of

_PAIRS = {2: ((0, 0), (0, 1), (1, 1)), 3: ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))}


@functools.lru_cache(maxsize=64)
def _reference_sums(p, bcs, ws):
    """(M (TD, TD, ldof, ldof), sum_q w_q phi_i phi_j) of the degree-p basis at
    the rule (points and weights as tuples of numbers), with
    M[a, b, i, j] = sum_q w_q R'_ia R'_jb, R' the reference gradients reduced by
    sum_m grad lambda_m = 0.  Formed on the host, so that a table is complete
    when it is uploaded, whichever stream or thread reads it first, and summed
    in extended precision: every cell multiplies the same table, whose rounding
    would not average out over the cells of a row."""
    bc, w = np.array(bcs), np.array(ws, dtype=np.longdouble)
    R = grad_shape_function(bc, p).astype(np.longdouble)
    R = (R[:, :, 1:] - R[:, :, :1]).transpose(0, 2, 1)                # (NQ, TD, ldof)
    phi = shape_function(bc, p).astype(np.longdouble)
    nq, td, ldof = R.shape
    F = np.ascontiguousarray(R).reshape(nq, -1)
    M = ((F * w[:, None]).T @ F).reshape(td, ldof, td, ldof).transpose(0, 2, 1, 3)
    return np.ascontiguousarray(M, dtype=np.float64), ((phi * w[:, None]).T @ phi).astype(np.float64)


def _sums(space, q):
    bcs, ws = space.mesh.quadrature_formula(q).get_quadrature_points_and_weights()
    return _reference_sums(space.p, tuple(map(tuple, bcs.tolist())), tuple(ws.tolist()))


def p1_table(space, q):
    """(NS + 1, TD + 1, TD + 1) table of fa_assemble_p1_rows, FP64, kept per rule."""
    cache = space.__dict__.setdefault('_row_tables', {})
    if q not in cache:
        M, mass = _sums(space, q)
        rows = [M[a, b] if a == b else M[a, b] + M[b, a] for a, b in _PAIRS[space.TD]]
        cache[q] = torch.as_tensor(np.stack(rows + [mass]), device=space.device)
    return cache[q]


def elasticity_table(scalar_space, q):
    """(TD, TD, ldof, ldof) table of fa_assemble_elasticity_rows, kept per rule."""
    cache = scalar_space.__dict__.setdefault('_elast_row_tables', {})
    if q not in cache:
        cache[q] = torch.as_tensor(_sums(scalar_space, q)[0], device=scalar_space.device)
    return cache[q]


def _wide_nodes(mesh, TD):
    rows = mesh.node_rows16()
    return rows if rows.shape[1] == (2 if TD == 2 else 4) else None


def p1_values(space, q, spec, pat, dtype):
    """CSR values of P1 diffusion and mass with coefficient specs `spec`
    ({'diff', 'mass'}, constant on each cell), or None when the mesh or
    pattern is not one of these kernels'."""
    mesh = space.mesh
    nodew = _wide_nodes(mesh, space.TD)
    pos = pat.row_positions()
    if nodew is None or pos is None:
        return None
    L = nat.lib()
    (dk, ds, dc), (mk, ms, mc) = spec['diff'], spec['mass']
    rec = nat.workspace(L.fa_p1_records_bytes(space.TD, pat.nc), space.device)
    values = torch.empty(pat.nnz, dtype=dtype, device=space.device)
    st = L.fa_assemble_p1_rows(nat.dtype_code(dtype), space.TD, pat.gdof, pat.nc, nat.ptr(nodew),
                               nat.ptr(space.cell_to_dof()), nat.ptr(p1_table(space, q)), dk, ds, nat.ptr(dc), mk, ms,
                               nat.ptr(mc), nat.ptr(pat.adj_ptr), nat.ptr(pat.adj), nat.ptr(pat.indptr), nat.ptr(pos),
                               pat.max_row, nat.ptr(rec), rec.numel(), nat.ptr(values), nat.stream())
    if st == nat.FA_ECAPACITY:
        return None
    nat.check(st, "fa_assemble_p1_rows")
    return values


# 3D vector spaces of at least this many scalar DOFs sum elasticity rows from a
# record per cell (2D ones always): below, the few waves' chains of incidences
# are longer than the element matrices take (8^3 cells at P2: 57 against 38 us;
# 40^3: 0.64 against 1.97 ms).  P4 tetrahedra keep the element matrices: the
# table's 88 KB of LDS leave two waves a CU (10^3: 528 against 483 us).
ELASTICITY_MIN_DOFS = 32768


def elasticity_values(space, it, dtype):
    """CSR values of a LinearElasticityIntegrator over all cells on the vector
    space's pattern, or None (see p1_values)."""
    ss = space.scalar_space
    mesh = ss.mesh
    if ss.TD == 3 and (ss.p > 3 or ss.number_of_global_dofs() < ELASTICITY_MIN_DOFS):
        return None
    pat = pattern_of(space)
    nodew = _wide_nodes(mesh, ss.TD)
    pos = pat.vector_positions(ss.TD, space.dof_priority)
    if nodew is None or pos is None:
        return None
    L = nat.lib()
    q = ss.p + 3 if it.q is None else it.q
    table = elasticity_table(ss, q)
    cell = mesh.cell.to(torch.int32).contiguous()
    cA, cB, cC, cD = it._coefficients(space.GD, space.dof_priority)
    rec = nat.workspace(L.fa_elasticity_records_bytes(ss.TD, pat.nc), space.device)
    values = torch.empty(pat.nnz, dtype=dtype, device=space.device)
    st = L.fa_assemble_elasticity_rows(nat.dtype_code(dtype), ss.TD, int(space.dof_priority),
                                       ss.number_of_global_dofs(), pat.nc, pat.ldof // ss.TD, nat.ptr(nodew),
                                       nat.ptr(cell), nat.ptr(table), cA, cB, cC, cD, nat.ptr(pat.adj_ptr),
                                       nat.ptr(pat.adj), nat.ptr(pat.indptr), pat.nnz, nat.ptr(pos), pat.max_row,
                                       nat.ptr(rec), rec.numel(), nat.ptr(values), nat.stream())
    if st == nat.FA_ECAPACITY:
        return None
    nat.check(st, "fa_assemble_elasticity_rows")
    return values
