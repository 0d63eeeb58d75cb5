"""CG on matrices that fit one workgroup's registers: at the edges of 8, 16, 24
and 32 entries per thread (8,192 to 32,768 entries), of one, two and four rows per
thread (1,024, 2,048, 4,096 rows) and one step beyond; a row that spans a hundred
threads; an empty row (the general path).  Against the same recurrence in numpy.

Bars: the diagonal dominates by 2, so |A^-1| |A| < 4 in the row-sum norm after
scaling and x agrees within 4 * sqrt(n) * 1e-11 of |x|; the iteration counts
within 1, as the residual shrinks at least threefold per iteration and rounding
decides the last one only.
"""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

import libmesh_amd as L

pytestmark = pytest.mark.gpu


def spd(rng, n, nnz):
    """n rows, n + 2 * ((nnz - n) // 2) entries, diagonally dominant"""
    pairs, seen = (nnz - n) // 2, set()
    while len(seen) < pairs:
        i, j = rng.integers(0, n, 2)
        if i != j:
            seen.add((max(i, j), min(i, j)))
    r, c = np.array(sorted(seen)).reshape(-1, 2).T
    w = rng.uniform(-1, 1, pairs)
    A = sp.coo_matrix((w, (r, c)), shape=(n, n))
    A = (A + A.T).tocsr()
    return dominant(rng, A)


def dominant(rng, A):
    A = A + sp.diags(3 * np.asarray(abs(A).sum(1)).ravel() + rng.uniform(1, 4, A.shape[0]))
    A = A.tocsr()
    A.sort_indices()
    return A


def arrow(rng, n, length):
    A = sp.lil_matrix((n, n))
    A[n // 2, :length] = rng.uniform(-1, 1, length)
    A[n // 2, n // 2] = 0
    A = A.tocsr()
    A.eliminate_zeros()
    return dominant(rng, A + A.T)


def reference(A, b, jacobi, rtol):
    d = 1 / A.diagonal() if jacobi else np.ones(len(b))
    x, r = np.zeros(len(b)), b.copy()
    p = d * r
    rz, its = r @ p, 0
    while True:
        q = A @ p
        a = rz / (p @ q)
        x += a * p
        r -= a * q
        if np.linalg.norm(r) < rtol * np.linalg.norm(b):
            return x, its
        its += 1
        new = r @ (d * r)
        p = d * r + new / rz * p
        rz = new


CASES = [(1, 1), (2, 4), (63, 700), (1024, 8192), (1025, 8193), (1023, 8195), (1024, 16384), (2048, 16386),
         (2049, 24575), (900, 24578), (4096, 32768), (1500, 32768), (4095, 32767), (4096, 32770), (4097, 20001)]


@pytest.mark.parametrize("what", CASES + ["arrow"], ids=str)
def test_small_cg(ctx, what):
    rng = np.random.default_rng(5)
    A = arrow(rng, 1100, 1000) if what == "arrow" else spd(rng, *what)
    n = A.shape[0]
    b = rng.standard_normal(n)
    rp, ci = A.indptr.astype(np.int32), A.indices.astype(np.int32)
    h = C.c_void_p()
    L.check(L.hip().lmh_matrix_create_csr(ctx.h, n, L._ptr(rp), L._ptr(ci), C.byref(h)))
    try:
        L.check(L.hip().lmh_matrix_set_values(h, L._ptr(A.data)))
        bd, x = L.DeviceArray(ctx, n, data=b), L.DeviceArray(ctx, n)
        for jacobi in (True, False):
            L.check(L.hip().lmh_matrix_set_preconditioner(h, L.PRECOND_JACOBI if jacobi else L.PRECOND_IDENTITY))
            ref, ref_its = reference(A, b, jacobi, 1e-11)
            got = []
            for solve in (L.hip().lmh_cg_solve, L.hip().lmh_cg_solve_noalloc):
                x.zero()
                its, res, why = C.c_int64(), C.c_double(), C.c_int()
                L.check(solve(h, bd.ptr, x.ptr, 1e-11, 5000, C.byref(its), C.byref(res), C.byref(why)))
                xh = x.download()
                assert why.value == L.CONVERGED_RTOL and abs(its.value - ref_its) <= 1
                assert np.linalg.norm(xh - ref) <= 4e-11 * np.sqrt(n) * np.linalg.norm(ref)
                got.append(xh)
            assert np.array_equal(*got)
            # stopped by the iteration limit, then resumed from there
            if ref_its > 3:
                x.zero()
                L.check(L.hip().lmh_cg_solve(h, bd.ptr, x.ptr, 1e-11, 3, C.byref(its), C.byref(res), C.byref(why)))
                assert why.value == L.DIVERGED_ITS and its.value == 3
                r = np.linalg.norm(b - A @ x.download()) / np.linalg.norm(b)
                assert abs(res.value - r) <= 1e-12 + 1e-9 * r
    finally:
        L.hip().lmh_matrix_destroy(h)


def test_empty_row(ctx):
    rng = np.random.default_rng(6)
    A = spd(rng, 300, 3000).tolil()
    A[77] = 0
    A[:, 77] = 0
    A = A.tocsr()
    A.eliminate_zeros()
    b = rng.standard_normal(300)
    b[77] = 0
    rp, ci = A.indptr.astype(np.int32), A.indices.astype(np.int32)
    h = C.c_void_p()
    L.check(L.hip().lmh_matrix_create_csr(ctx.h, 300, L._ptr(rp), L._ptr(ci), C.byref(h)))
    try:
        L.check(L.hip().lmh_matrix_set_values(h, L._ptr(A.data)))
        L.check(L.hip().lmh_matrix_set_preconditioner(h, L.PRECOND_IDENTITY))
        ref, ref_its = reference(A, b, False, 1e-11)
        bd, x = L.DeviceArray(ctx, 300, data=b), L.DeviceArray(ctx, 300)
        x.zero()
        its, res, why = C.c_int64(), C.c_double(), C.c_int()
        L.check(L.hip().lmh_cg_solve(h, bd.ptr, x.ptr, 1e-11, 500, C.byref(its), C.byref(res), C.byref(why)))
        assert why.value == L.CONVERGED_RTOL and abs(its.value - ref_its) <= 1
        assert np.linalg.norm(x.download() - ref) <= 4e-11 * np.sqrt(300) * np.linalg.norm(ref)
    finally:
        L.hip().lmh_matrix_destroy(h)


@pytest.mark.parametrize("n,length", [(2100, 2048), (4096, 4096)])
def test_longest_rows(ctx, n, length):
    """A row over 256 threads of the workgroup, whose pieces its owner adds alone"""
    rng = np.random.default_rng(7)
    A = arrow(rng, n, length)
    b = rng.standard_normal(n)
    rp, ci = A.indptr.astype(np.int32), A.indices.astype(np.int32)
    h = C.c_void_p()
    L.check(L.hip().lmh_matrix_create_csr(ctx.h, n, L._ptr(rp), L._ptr(ci), C.byref(h)))
    try:
        L.check(L.hip().lmh_matrix_set_values(h, L._ptr(A.data)))
        ref, ref_its = reference(A, b, True, 1e-11)
        bd, x = L.DeviceArray(ctx, n, data=b), L.DeviceArray(ctx, n)
        x.zero()
        its, res, why = C.c_int64(), C.c_double(), C.c_int()
        ctx.profile_reset()
        ctx.profile(True)
        L.check(L.hip().lmh_cg_solve(h, bd.ptr, x.ptr, 1e-11, 5000, C.byref(its), C.byref(res), C.byref(why)))
        ctx.profile(False)
        assert ctx.profile_query("cg_small")[1] == 1
        assert why.value == L.CONVERGED_RTOL and abs(its.value - ref_its) <= 1
        assert np.linalg.norm(x.download() - ref) <= 4e-11 * np.sqrt(n) * np.linalg.norm(ref)
    finally:
        L.hip().lmh_matrix_destroy(h)
