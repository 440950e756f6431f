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


def _rule(space, q):
    """Points and weights of rule q as tuples of numbers."""
    bcs, ws = space.mesh.quadrature_formula(q).get_quadrature_points_and_weights()
    return tuple(map(tuple, bcs.tolist())), tuple(ws.tolist())


@functools.lru_cache(maxsize=64)
def _p1_sums(bcs, ws):
    """Table of fa_assemble_p1_rows for the rule, formed on the host: complete when it is uploaded, whichever
    stream or thread reads it first, and summed in extended precision, since
    every cell multiplies the same table and its rounding would not average out
    over the cells of a row (2.26M tetrahedra: 3.2e-16 off 64 bits summed in
    FP64, 2.5e-16 so)."""
    bc, w = np.array(bcs), np.array(ws, dtype=np.longdouble)
    R = grad_shape_function(bc, 1).astype(np.longdouble)
    R = R[:, :, 1:] - R[:, :, :1]                                     # sum_m grad lambda_m = 0
    phi = shape_function(bc, 1).astype(np.longdouble)
    M = np.einsum('q, qia, qjb -> abij', w, R, R)
    rows = [M[a, b] if a == b else M[a, b] + M[b, a] for a, b in _PAIRS[R.shape[2]]]
    return np.stack(rows + [np.einsum('q, qi, qj -> ij', w, phi, phi)]).astype(np.float64)


def p1_table(space, q):
    """(NS + 1, TD + 1, TD + 1) table of fa_assemble_p1_rows, FP64, kept per rule."""
    cache = space.__dict__.setdefault('_row_tables', {})
    if q not in cache:
        cache[q] = torch.as_tensor(_p1_sums(*_rule(space, q)), device=space.device)
    return cache[q]


@functools.lru_cache(maxsize=64)
def _elasticity_tables(device, p, bcs, ws):
    """(M (ldof, ldof, TD + 1, TD + 1), reduced (TD, TD, ldof, ldof)) of the
    degree-p basis at the rule, FP64 on the device and complete there before any
    other stream or thread can see them:
    M[i, j, m, n] = sum_q w_q R[q, i, m] R[q, j, n], and M reduced by
    sum_m grad lambda_m = 0.  Rows and element matrices share M's roundings
    (against 64 bits, P2 triangles 200^2: 1.4e-16; 2.2e-16 where the rows had a
    sum of reduced gradients of their own)."""
    R = torch.as_tensor(grad_shape_function(np.array(bcs), p), device=device)
    M = torch.einsum('q, qim, qjn -> ijmn', torch.as_tensor(np.array(ws), device=device), R, R).contiguous()
    V = M.permute(2, 3, 0, 1)
    reduced = (V[1:, 1:] - V[:1, 1:] - V[1:, :1] + V[:1, :1]).contiguous()
    if M.is_cuda:
        torch.cuda.current_stream(device).synchronize()
    return M, reduced


def elasticity_tables(scalar_space, q):
    """_elasticity_tables of a scalar space's rule: M for fa_element_elasticity,
    reduced for fa_assemble_elasticity_rows."""
    cache = scalar_space.__dict__.setdefault('_elast_tables', {})
    if q not in cache:
        cache[q] = _elasticity_tables(scalar_space.device, scalar_space.p, *_rule(scalar_space, q))
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
    table = elasticity_tables(ss, q)[1]
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
