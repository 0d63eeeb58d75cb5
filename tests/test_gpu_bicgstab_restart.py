"""BiCGSTAB where its denominators vanish.  r becomes exactly orthogonal to r0: copies of a 3 x 3 block
whose first iteration, in whole numbers up to the weight w, ends with (r0, r) = 0.
With w = 3/5 the loop restarts, as the oracle's restatement of Eigen's does, and
solves the system; with w = 0 that loop would divide by it, and the solve reports
a breakdown.  3 to 30,000 rows: one workgroup of vector sums to many, with and
without windows.

An upper bidiagonal matrix whose Krylov space is nearly used up after two
iterations, so that (r0, r) and (r0, v) are rounding and the order of the sums
decides whether one is exactly 0: it must converge in any order, here that of
every grid.

Bars: the oracle's count (from 0 after the restart) within 2 for the blocks; x
within 1e-9 of A^-1 b (cond(A) < 10 and |r| <= 1e-10 |b|)."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

import libmesh_amd as L
import oracle as O

pytestmark = pytest.mark.gpu

RESTART = np.array([[1.0, 1, 1], [1, 2, 0], [-1, 0, 1]])
STUCK = np.array([[1.0, 1, 1], [1, 1, 0], [-1, 2, 1]])


def blocks(block, copies):
    A = sp.block_diag([block] * copies, format="csr")
    A.eliminate_zeros()
    return A, np.tile([1.0, 0, 0], copies)


def solve(ctx, A, b, windows=1, maxits=100, identity=True):
    n = len(b)
    rp, ci = A.indptr.astype(np.int32), A.indices.astype(np.int32)
    h = C.c_void_p()
    L.check(L.hip().lmh_matrix_create_csr(ctx.h, n, L._ptr(rp), L._ptr(ci), C.byref(h)))
    try:
        L.check(L.hip().lmh_matrix_set_values(h, L._ptr(A.data)))
        L.check(L.hip().lmh_matrix_set_preconditioner(h, L.PRECOND_IDENTITY if identity else L.PRECOND_JACOBI))
        L.check(L.hip().lmh_matrix_set_fp32_compression(h, windows))
        bd, x = L.DeviceArray(ctx, n, data=b), L.DeviceArray(ctx, n)
        x.zero()
        its, res, why = C.c_int64(), C.c_double(), C.c_int()
        L.check(L.hip().lmh_bicgstab_solve(h, bd.ptr, x.ptr, 1e-10, maxits, C.byref(its), C.byref(res), C.byref(why)))
        return x.download(), its.value, res.value, why.value
    finally:
        L.hip().lmh_matrix_destroy(h)


@pytest.mark.parametrize("windows", [1, 0])
@pytest.mark.parametrize("copies", [1, 100, 3000, 10000])
def test_restart(ctx, copies, windows):
    A, b = blocks(RESTART, copies)
    x, its, res, why = solve(ctx, A, b, windows)
    ox, oits, _ = O.bicgstab_eigen(A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data, b, 1e-10, 100,
                                   precond="identity")
    exact = np.tile(np.linalg.solve(RESTART, [1.0, 0, 0]), copies)
    assert np.abs(ox - exact).max() < 1e-9
    assert why == L.CONVERGED_RTOL and res <= 1e-10 and abs(its - oits) <= 2
    assert np.abs(x - exact).max() < 1e-9


def test_limit_counts_all_iterations(ctx):
    _, its, res, why = solve(ctx, *blocks(RESTART, 100), maxits=2)
    assert why == L.DIVERGED_ITS and its == 2 and res > 1e-10


@pytest.mark.parametrize("copies", [1, 3000])
def test_breakdown(ctx, copies):
    assert solve(ctx, *blocks(STUCK, copies))[3] == L.DIVERGED_BREAKDOWN


@pytest.mark.parametrize("identity", [True, False])
@pytest.mark.parametrize("n", [7, 33, 64, 100, 511, 513, 1500, 3000, 9000, 16383, 16384, 40000])
def test_any_order_converges(ctx, n, identity):
    A = sp.diags([np.ones(n - 1), 4.0 * np.ones(n)], [1, 0], format="csr")
    for windows in (1, 0):
        x, _, res, why = solve(ctx, A, np.ones(n), windows, identity=identity)
        assert why == L.CONVERGED_RTOL and res <= 1e-10
        exact = np.empty(n)
        exact[-1] = 0.25
        for i in range(n - 2, -1, -1):
            exact[i] = 0.25 * (1.0 - exact[i + 1])
        assert np.abs(x - exact).max() < 1e-9 * np.sqrt(n)
