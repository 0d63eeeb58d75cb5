"""A mixed solve that ends at its iteration limit reports the residual of the x it
returns, whatever the product's time: |b - A x| / |b| formed on the host, to the
rounding of the product (1e-12 of |A| |x| / |b|, the rows summing at most 2,001
entries)."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

import libmesh_amd as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(300, 3), (3000, 1000), (200000, 30)])
def test_reported_residual(ctx, n, k):
    rng = np.random.default_rng(17)
    A = sp.diags([rng.uniform(-1, 1) * np.ones(n - d) for d in range(1, k + 1)], list(range(1, k + 1)), format="csr")
    A = A + A.T
    A = (A + sp.diags(np.asarray(abs(A).sum(1)).ravel() + 1.0)).tocsr()
    A.sort_indices()
    rp, ci, v = A.indptr.astype(np.int32), A.indices.astype(np.int32), np.ascontiguousarray(A.data)
    h = C.c_void_p()
    L.check(L.hip().lmh_matrix_create_csr(ctx.h, n, L._ptr(rp), L._ptr(ci), C.byref(h)))
    try:
        L.check(L.hip().lmh_matrix_set_values(h, L._ptr(v)))
        L.check(L.hip().lmh_matrix_make_fp32(h))
        bh = rng.standard_normal(n)
        b, x = L.DeviceArray(ctx, n, data=bh), L.DeviceArray(ctx, n)
        its, res, why, stats = C.c_int64(), C.c_double(), C.c_int(), np.zeros(3)
        for limit in (1, 2, 3, 1, 2, 3):
            x.zero()
            L.check(L.hip().lmh_mixed_solve(h, b.ptr, x.ptr, 1e-10, 0.1, 0, limit, C.byref(its), C.byref(res),
                                            C.byref(why), L._ptr(stats)))
            xh = x.download()
            true = np.linalg.norm(bh - A @ xh) / np.linalg.norm(bh)
            bar = 1e-12 * np.linalg.norm(abs(A) @ abs(xh)) / np.linalg.norm(bh)
            assert why.value == L.DIVERGED_ITS and abs(res.value - true) <= bar and stats[2] == res.value, limit
    finally:
        L.hip().lmh_matrix_destroy(h)
