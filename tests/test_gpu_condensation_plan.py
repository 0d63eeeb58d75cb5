"""Condensation refreshes over every form a plan can take: condensed rows longer
than 32 entries, rows beyond 255 columns (16-bit places), structural couplings
between condensed DoFs that hold zeros, and the rows no plan takes (more than 32
condensed columns, longer than a row block).  First values and refreshed values,
forward and backward steps against scipy's A_uu - A_uc D^-1 A_cu.

Bars: an entry is one value and at most 45 subtractions of a product and a
quotient: within 50 * 4 * 1.2e-16 < 3e-14 of the sum of the terms' absolute values;
the steps sum at most 2,100 such terms: within 2,200 * 4 * 1.2e-16 < 1.1e-12.
"""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

import libmesh_amd as L

pytestmark = pytest.mark.gpu

# reduced DoFs, condensed DoFs, columns of a condensed row, window they are drawn from
FORMS = {"small": (300, 60, 12, 40), "one": (9, 1, 9, 9), "long": (500, 40, 45, 60), "wide": (900, 12, 290, 320),
         "many": (400, 45, 20, 50), "huge": (2200, 2, 2100, 2200), "coupled": (300, 60, 12, 40)}


def build(name):
    rng = np.random.default_rng(9)
    nr, nc, size, window = FORMS[name]
    n = nr + nc
    perm = rng.permutation(n)  # condensed DoFs anywhere in the numbering
    red, cond = np.sort(perm[:nr]), np.sort(perm[nr:])
    pairs = [np.stack([red, red])]
    for q, c in enumerate(cond):
        lo = 0 if name == "many" else rng.integers(0, nr - window + 1)
        cols = red[lo + rng.permutation(window)[:size]]
        if name == "many":
            cols[0] = red[3]  # one row with every condensed column
            cols = np.unique(cols)
        full = np.append(cols, c)
        pairs.append(np.stack(np.meshgrid(full, full)).reshape(2, -1))
        if name == "coupled" and q:
            pairs.append(np.array([[c, cond[q - 1]], [cond[q - 1], c]]))
    r, c = np.concatenate(pairs, axis=1)
    A = sp.csr_matrix((np.ones(r.size), (r, c)), shape=(n, n))
    A.sort_indices()
    return A, red, cond, rng


def values(A, cond, rng):
    v = rng.uniform(-1, 1, A.nnz)
    v[rng.random(A.nnz) < 0.1] = 0.0  # some couplings vanish
    rows = np.repeat(np.arange(A.shape[0]), np.diff(A.indptr))
    isc = np.zeros(A.shape[0], bool)
    isc[cond] = True
    v[isc[rows] & isc[A.indices] & (rows != A.indices)] = 0.0
    v[(rows == A.indices) & isc[rows]] = rng.uniform(1, 3, cond.size) * rng.choice([-1, 1], cond.size)
    return v


@pytest.mark.parametrize("name", FORMS)
def test_plan_forms(ctx, name):
    A, red, cond, rng = build(name)
    n = A.shape[0]
    rp, ci = A.indptr.astype(np.int32), A.indices.astype(np.int32)
    h, sc = C.c_void_p(), C.c_void_p()
    L.check(L.hip().lmh_matrix_create_csr(ctx.h, n, L._ptr(rp), L._ptr(ci), C.byref(h)))
    try:
        cd = cond.astype(np.int32)
        for refresh in range(3):
            A.data = values(A, cond, rng)
            L.check(L.hip().lmh_matrix_set_values(h, L._ptr(A.data)))
            if refresh == 0:
                L.check(L.hip().lmh_condensation_create(h, cd.size, L._ptr(cd), C.byref(sc)))
                R = C.c_void_p(L.hip().lmh_condensation_reduced_matrix(sc))
                nnz = L.hip().lmh_matrix_nnz(R)
                srp, sci = np.empty(red.size + 1, np.int32), np.empty(nnz, np.int32)
                L.check(L.hip().lmh_matrix_get_pattern(R, L._ptr(srp), L._ptr(sci)))
            else:
                L.check(L.hip().lmh_condensation_setup(sc))
            v = np.empty(nnz)
            L.check(L.hip().lmh_matrix_get_values(R, L._ptr(v)))
            S = sp.csr_matrix((v, sci, srp), shape=(red.size,) * 2)
            Auu, Auc, Acu = A[red][:, red], A[red][:, cond], A[cond][:, red]
            D = A.diagonal()[cond]
            ref = Auu - Auc @ sp.diags(1 / D) @ Acu
            size = abs(Auu) + abs(Auc) @ sp.diags(1 / abs(D)) @ abs(Acu)
            assert (abs(S - ref) > 3e-14 * size).nnz == 0
            b, y = rng.standard_normal(n), rng.standard_normal(red.size)
            bd, yd = L.DeviceArray(ctx, n, data=b), L.DeviceArray(ctx, red.size, data=y)
            gd, xd = L.DeviceArray(ctx, red.size), L.DeviceArray(ctx, n)
            L.check(L.hip().lmh_condensation_forward(sc, bd.ptr, gd.ptr))
            L.check(L.hip().lmh_condensation_backward(sc, bd.ptr, yd.ptr, xd.ptr))
            fs = abs(b[red]) + abs(Auc) @ abs(b[cond] / D)
            assert np.all(abs(gd.download() - (b[red] - Auc @ (b[cond] / D))) <= 1.1e-12 * fs)
            x = xd.download()
            assert np.array_equal(x[red], y)
            bs = (abs(b[cond]) + abs(Acu) @ abs(y)) / abs(D)
            assert np.all(abs(x[cond] - (b[cond] - Acu @ y) / D) <= 1.1e-12 * bs)
        # a vanishing pivot is refused at a refresh, and the next good values are taken
        good = A.data.copy()
        k = rp[cond[-1]] + np.searchsorted(ci[rp[cond[-1]]:rp[cond[-1] + 1]], cond[-1])
        A.data[k] = 0.0
        L.check(L.hip().lmh_matrix_set_values(h, L._ptr(A.data)))
        with pytest.raises(L.LmhError, match="zero diagonal"):
            L.check(L.hip().lmh_condensation_setup(sc))
        if name == "coupled":
            A.data = good.copy()
            k = rp[cond[1]] + np.searchsorted(ci[rp[cond[1]]:rp[cond[1] + 1]], cond[0])
            A.data[k] = 0.5
            L.check(L.hip().lmh_matrix_set_values(h, L._ptr(A.data)))
            with pytest.raises(L.LmhError, match="couple"):
                L.check(L.hip().lmh_condensation_setup(sc))
        L.check(L.hip().lmh_matrix_set_values(h, L._ptr(good)))
        L.check(L.hip().lmh_condensation_setup(sc))
        w = np.empty(nnz)
        L.check(L.hip().lmh_matrix_get_values(R, L._ptr(w)))
        assert np.array_equal(w, v)
    finally:
        if sc.value:
            L.hip().lmh_condensation_destroy(sc)
        L.hip().lmh_matrix_destroy(h)
