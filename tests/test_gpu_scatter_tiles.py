"""The gather scatter on row tiles: CSR values and right-hand side summed in
ascending element order, bit for bit the sequential sum, for element DoF counts
of every lane grouping (4, 8, 10, 12, 24, 27, 30), one to many tiles, and the
row-at-a-time kernel beyond 32 DoFs (81)."""
import numpy as np
import pytest

import libmesh_amd as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t,nv,box", [
    (L.HEX27, 1, (1, 1, 1)), (L.HEX27, 1, (5, 4, 3)), (L.HEX8, 1, (9, 7, 5)), (L.HEX8, 3, (4, 3, 5)),
    (L.TET4, 1, (1, 1, 1)), (L.TET4, 1, (4, 5, 3)), (L.TET4, 3, (3, 2, 2)), (L.TET10, 1, (1, 1, 1)),
    (L.TET10, 1, (3, 2, 4)), (L.TET10, 3, (2, 1, 2)), (L.HEX27, 3, (2, 2, 2)), (L.HEX27, 1, (17, 16, 15))])
def test_scatter_is_the_sequential_sum(ctx, t, nv, box):
    p = L.Problem(box[0], t, nv, L.ALL_FACES, box[1], box[2])
    g = L.GpuProblem.from_problem(ctx, p)
    rng = np.random.default_rng(29)
    Ke = rng.standard_normal((p.n_elem, p.dpe, p.dpe))
    Fe = rng.standard_normal((p.n_elem, p.dpe))
    Kd, Fd = L.DeviceArray(ctx, Ke.size, data=Ke.ravel()), L.DeviceArray(ctx, Fe.size, data=Fe.ravel())
    R = L.DeviceArray(ctx, p.n_dofs, data=rng.standard_normal(p.n_dofs))  # overwritten
    g.set_values(rng.standard_normal(g.nnz))
    L.check(L.hip().lmh_matrix_scatter_elements(g.matrix, Kd.ptr, Fd.ptr, R.ptr))
    rp, ci = g.pattern()
    d = p.elem_dofs.astype(np.int64)
    key = (d[:, :, None] * p.n_dofs + d[:, None, :]).ravel()
    entry = np.repeat(np.arange(p.n_dofs, dtype=np.int64), np.diff(rp)) * p.n_dofs + ci
    vals, rhs = np.zeros(g.nnz), np.zeros(p.n_dofs)
    np.add.at(vals, np.searchsorted(entry, key), Ke.ravel())  # one at a time, in element order
    np.add.at(rhs, d.ravel(), Fe.ravel())
    assert np.array_equal(g.values(), vals)
    assert np.array_equal(R.download(), rhs)
    # without a right-hand side, and the vector alone
    g.set_values(np.zeros(g.nnz))
    L.check(L.hip().lmh_matrix_scatter_elements(g.matrix, Kd.ptr, None, None))
    assert np.array_equal(g.values(), vals)
    R.zero()
    L.check(L.hip().lmh_matrix_scatter_elements(g.matrix, None, Fd.ptr, R.ptr))
    assert np.array_equal(R.download(), rhs)
    g.close()


@pytest.mark.parametrize("t,nv,box", [
    (L.HEX8, 1, (11, 11, 11)), (L.HEX8, 1, (12, 12, 12)), (L.HEX27, 1, (13, 13, 13)), (L.HEX27, 1, (15, 15, 15)),
    (L.TET4, 1, (10, 10, 9)), (L.TET4, 1, (10, 10, 10)), (L.TET10, 1, (5, 5, 5)), (L.TET10, 1, (6, 5, 5)),
    (L.TET4, 3, (7, 6, 6)), (L.TET4, 3, (7, 7, 7)), (L.TET10, 3, (3, 3, 4)), (L.TET10, 3, (4, 4, 3))])
def test_both_ways_to_the_plan(ctx, t, nv, box):
    """On each side of the size to which the plan is made in one launch (hexahedra), and
    of the one from which tetrahedral matrices have a plan (5,500 rows)"""
    test_scatter_is_the_sequential_sum(ctx, t, nv, box)
