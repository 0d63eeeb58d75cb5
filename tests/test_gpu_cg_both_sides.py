"""CG's special ends on both implementations: the kernel that holds a small matrix
on one workgroup (Q2 2^3: 125 rows) and the three kernels an iteration (Q2 4^3: 35,937
entries, over its limit).  Zero right-hand side, NaN and Inf, a zero operator, the
iteration limit; and the allocation-free solve of a small and of a larger system
on scratch that holds a larger one's vectors, first and second."""
import numpy as np
import pytest

import libmesh_amd as L
from test_zz_no_alloc import solve_both

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[2, 4])
def system(ctx, request):
    n = request.param
    p = L.Problem(n, L.HEX27)
    g = L.GpuProblem.from_problem(ctx, p)
    b = L.DeviceArray(ctx, p.n_dofs)
    g.assemble_poisson(3, None, 1, b)
    yield ctx, n, p, g, b, L.DeviceArray(ctx, p.n_dofs)
    g.close()


def test_the_kernel_that_runs(system):
    ctx, n, p, g, b, x = system
    x.zero()
    ctx.profile_reset()
    ctx.profile(True)
    its, res, why = g.cg(b, x, 1e-10, 100)
    ctx.profile(False)
    assert why == L.CONVERGED_RTOL
    assert (ctx.profile_query("cg_small")[1] == 1) == (n == 2)
    assert (ctx.profile_query("cg_spmv_fp64")[1] > 0) == (n == 4)


def test_zero_rhs(system):
    ctx, n, p, g, b, x = system
    z = L.DeviceArray(ctx, p.n_dofs)
    z.zero()
    for solve in (g.cg, g.cg_noalloc):
        x.upload(np.random.default_rng(0).standard_normal(p.n_dofs))
        its, res, why = solve(z, x, 1e-10, 100)
        assert its == 0 and why == L.CONVERGED_RTOL and res == 0.0
        assert not x.download().any()


def test_failure_reasons(system):
    ctx, n, p, g, b, x = system
    for solve in (g.cg, g.cg_noalloc):
        x.zero()
        its, res, why = solve(b, x, 1e-14, 2)
        assert its == 2 and why == L.DIVERGED_ITS and res > 1e-14
        for bad in (np.nan, np.inf, -np.inf):
            bh = b.download()
            bh[p.n_dofs // 2] = bad
            bn = L.DeviceArray(ctx, p.n_dofs, data=bh)
            x.zero()
            its, res, why = solve(bn, x, 1e-10, 100)
            assert why == L.DIVERGED_NANORINF and its == 0, bad
            bn.free()
    v = g.values()
    g.set_values(np.zeros(g.nnz))
    for solve in (g.cg, g.cg_noalloc):
        x.zero()
        assert solve(b, x, 1e-10, 100)[2] == L.DIVERGED_BREAKDOWN
    # a NaN in the operator comes up in the first product
    v[g.nnz // 2] = np.nan
    g.set_values(v)
    for solve in (g.cg, g.cg_noalloc):
        x.upload(np.ones(p.n_dofs))
        assert solve(b, x, 1e-10, 100)[2] == L.DIVERGED_NANORINF


@pytest.mark.parametrize("first", [True, False])
def test_noalloc_after_a_larger_system(ctx, first):
    for n, t, npts in ((8, L.HEX27, 3), (12, L.HEX8, 2), (5, L.HEX8, 2)):  # the second: 50,653 entries
        _, g, *_ = solve_both(ctx, n, t, npts, 0x5EED0400 + n, first)
        g.close()
