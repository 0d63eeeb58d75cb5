"""The batch's two row paths: DoFs in node blocks (3B, 3B + 1, 3B + 2 on one node)
and any other numbering, which takes the general row kernel.

Bars: against the FP64 oracle as in test_gpu_batch.py (values 2e-6 of the largest,
rhs 1e-12); between the paths the same element matrices are added in the same
order, so HEX8, HEX27 and TET10 agree to the bit; TET4 sums its rule before the
products in one path and after them in the other: 5 terms of FP32 rounding, within
2e-6.
"""
import numpy as np
import pytest
import scipy.sparse as sp

import libmesh_amd as L
import oracle as O

pytestmark = pytest.mark.gpu

NPTS = {L.HEX8: 2, L.HEX27: 3, L.TET4: 3, L.TET10: 5}
CLAMP = 1 << 4
SPECS = [(5, L.HEX8), (3, L.HEX27), (3, L.TET4), (2, L.TET10), (1, L.HEX27), (1, L.TET4), (12, L.HEX8)]


def renumber(name, n):
    d = np.arange(n)
    if name == "variables":
        return (d % 3) * (n // 3) + d // 3
    if name == "shifted":  # consecutive, but not from a multiple of three
        return (d + 1) % n
    if name == "nodes":  # node blocks in another order
        return np.random.default_rng(3).permutation(n // 3)[d // 3] * 3 + d % 3
    return d


@pytest.mark.parametrize("name", ["variables", "shifted", "nodes"])
def test_numberings_agree(ctx, name):
    probs = []
    for k, (n, t) in enumerate(SPECS):
        p = L.Problem(n, t, 3, CLAMP)
        p.perturb(11 + k, 0.2 if t in (L.HEX8, L.HEX27) else 0.1)
        probs.append(p)
    gps, perms = [], []
    for p in probs:
        for how in ("as built", name):
            f = renumber(how, p.n_dofs)
            cons = np.zeros_like(p.constrained)
            cons[f] = p.constrained
            gps.append(L.GpuProblem(ctx, p.coords, p.conn, p.elem_type, f[p.elem_dofs].astype(np.int32), p.n_dofs,
                                    cons, 3, build_matrix=False))
            perms.append(f)
    b = L.Batch(ctx, gps)
    for _ in range(2):
        b.assemble(1.0, 0.3, -1.0)
    for k, p in enumerate(probs):
        m = O.Mesh(*SPECS[k])
        m.perturb(11 + k, 0.2 if p.elem_type in (L.HEX8, L.HEX27) else 0.1)
        s = O.System(m, 3, CLAMP)
        vals, rhs = s.assemble_elasticity(NPTS[p.elem_type], 1.0, 0.3, -1.0)
        rp, ci = s.pattern()
        ref = sp.csr_matrix((vals, ci, rp), shape=(p.n_dofs,) * 2)
        dense = []
        for j in (2 * k, 2 * k + 1):
            f = perms[j]
            A = sp.csr_matrix((b.values(j), *b.pattern(j)[::-1]), shape=ref.shape)[f][:, f]
            A.sort_indices()
            assert np.array_equal(A.indices, ci) and np.array_equal(A.indptr, rp)
            assert np.abs(A.data - vals).max() < 2e-6 * np.abs(vals).max()
            assert np.abs(b.rhs(j)[f] - rhs).max() <= 1e-12 * np.abs(rhs).max()
            dense.append(A.data)
        if p.elem_type != L.TET4:
            assert np.array_equal(*dense)
    b.close()
