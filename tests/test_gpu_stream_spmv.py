"""Products on the streamed row blocks in every form the matrix can take:
8-bit windows, 16-bit windows (a row with more than 256 columns), blocks that
fit neither (int32 columns on the general kernel), empty rows, more rows in a
block than threads, a single row.  FP64 and FP32, windows on and off, against
scipy and bit for bit against each other.

Bars: a row sums at most 1,500 products, eight lanes of at most 190 and a tree;
FP64 within 1,500 * 1.2e-16 < 2e-13 of the row's absolute sum, FP32 within
1,500 * 6e-8 + 2 roundings of the inputs < 1.2e-4 of it.
"""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg

import libmesh_amd as L

pytestmark = pytest.mark.gpu


def banded(rng, n, per, width):
    cols = np.clip(np.arange(n)[:, None] + rng.integers(-width, width + 1, (n, per)), 0, n - 1)
    rows = np.repeat(np.arange(n), per)
    A = sp.csr_matrix((rng.standard_normal(rows.size), (rows, cols.ravel())), shape=(n, n))
    return (A + sp.diags(np.full(n, 4.0 * per))).tocsr()


def shape(name, rng):
    if name == "one":
        return sp.csr_matrix(np.array([[3.0]])), 8
    if name == "diagonal":  # 1016 rows per block
        return sp.diags(rng.uniform(1, 2, 5000), format="csr"), 0
    if name == "banded":
        return banded(rng, 4000, 30, 40), 8
    if name == "empty":  # rows without entries in the middle and at the end
        A = banded(rng, 3000, 20, 30).tolil()
        A[500:900] = 0
        A[2900:] = 0
        A = A.tocsr()
        A.eliminate_zeros()
        return A, 8
    if name == "wide_row":  # one row with 700 columns: 16-bit windows
        A = banded(rng, 3000, 25, 30).tolil()
        A[1200, 1000:1700] = 0.5
        return A.tocsr(), 16
    if name == "scattered":  # blocks split by rows until their windows fit
        return banded(rng, 4000, 20, 3999), 8
    A = banded(rng, 4000, 20, 50).tolil()  # one row with more than 768 columns: no windows
    A[77, rng.permutation(4000)[:1500]] = 0.25
    return A.tocsr(), 0


@pytest.mark.parametrize("name", ["one", "diagonal", "banded", "empty", "wide_row", "scattered", "long_row"])
def test_products(ctx, name):
    rng = np.random.default_rng(17)
    A, bits = shape(name, rng)
    A.sort_indices()
    n = A.shape[0]
    rp, ci = A.indptr.astype(np.int32), A.indices.astype(np.int32)
    h = C.c_void_p()
    L.check(L.hip().lmh_matrix_create_csr(ctx.h, n, L._ptr(rp), L._ptr(ci), C.byref(h)))
    try:
        L.check(L.hip().lmh_matrix_set_values(h, L._ptr(A.data)))
        L.check(L.hip().lmh_matrix_make_fp32(h))
        if name != "diagonal":
            assert L.hip().lmh_matrix_window_bits(h) == bits
        xh, bh = rng.standard_normal(n), rng.standard_normal(n)
        x, b = L.DeviceArray(ctx, n, data=xh), L.DeviceArray(ctx, n, data=bh)
        x32 = L.DeviceArray(ctx, n, np.float32, data=xh)
        y, r, y32 = L.DeviceArray(ctx, n), L.DeviceArray(ctx, n), L.DeviceArray(ctx, n, np.float32)
        got = []
        for on in (1, 0):
            L.check(L.hip().lmh_matrix_set_fp32_compression(h, on))
            L.check(L.hip().lmh_spmv(h, x.ptr, y.ptr))
            L.check(L.hip().lmh_residual(h, b.ptr, x.ptr, r.ptr))
            L.check(L.hip().lmh_spmv_fp32(h, x32.ptr, y32.ptr))
            got.append((y.download(), r.download(), y32.download()))
        for on, off in zip(*got):
            assert np.array_equal(on, off)
        scale = abs(A) @ np.abs(xh) + 1e-300
        assert np.all(np.abs(got[0][0] - A @ xh) <= 2e-13 * scale)
        assert np.all(np.abs(got[0][1] - (bh - A @ xh)) <= 2e-13 * (scale + np.abs(bh)))
        assert np.all(np.abs(got[0][2] - A @ xh) <= 1.2e-4 * scale)
    finally:
        L.hip().lmh_matrix_destroy(h)


@pytest.mark.parametrize("name", ["banded", "wide_row", "long_row"])
def test_solvers_agree_with_windows_on_and_off(ctx, name):
    """BiCGSTAB on a diagonally dominant matrix: the same row blocks and sums
    with the windows on and off, so the same iterates bit for bit."""
    rng = np.random.default_rng(23)
    A, _ = shape(name, rng)
    A.sort_indices()
    n = A.shape[0]
    rp, ci = A.indptr.astype(np.int32), A.indices.astype(np.int32)
    h = C.c_void_p()
    L.check(L.hip().lmh_matrix_create_csr(ctx.h, n, L._ptr(rp), L._ptr(ci), C.byref(h)))
    try:
        L.check(L.hip().lmh_matrix_set_values(h, L._ptr(A.data)))
        b, x = L.DeviceArray(ctx, n, data=rng.standard_normal(n)), L.DeviceArray(ctx, n)
        out = []
        for on in (1, 0):
            L.check(L.hip().lmh_matrix_set_fp32_compression(h, on))
            x.zero()
            its, res, reason = C.c_int64(), C.c_double(), C.c_int()
            L.check(L.hip().lmh_bicgstab_solve(h, b.ptr, x.ptr, 1e-12, 500, C.byref(its), C.byref(res),
                                               C.byref(reason)))
            assert reason.value == L.CONVERGED_RTOL
            out.append((its.value, x.download()))
        assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
        ref = sp.linalg.spsolve(A.tocsc(), b.download())
        assert np.linalg.norm(out[0][1] - ref) <= 1e-9 * np.linalg.norm(ref)
    finally:
        L.hip().lmh_matrix_destroy(h)
