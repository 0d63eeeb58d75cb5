"""GPU parity of the element kernels at the edges of their work split, against
the CPU oracle: residual, QoI derivative and adjoint gradient without an
element matrix (HEX27: seven elements per wavefront; TET4, TET10, HEX8: one
element per thread, 64 per workgroup) and the element matrices, all quadrature
rules they accept.

Bar 1e-12 normwise (max|a - b| / max|b|), as for the other FP64 element
results: an entry sums at most 27 points x 27 nodes x 9 products, so its
rounding is below a few hundred ulps (1e-13) of the largest entry.
"""
import numpy as np
import pytest

import libmesh_amd as L
import oracle as O

pytestmark = pytest.mark.gpu

SEED = 0x5EED0011


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


def problem(ctx, t, box):
    p = L.Problem(box[0], t, 1, L.ALL_FACES, box[1], box[2])
    m = O.Mesh(box[0], t, box[1], box[2])
    frac = 0.2 if t in (L.HEX8, L.HEX27) else 0.02
    p.perturb(SEED, frac)
    m.perturb(SEED, frac)
    return p, O.System(m), L.lognormal(p.n_elem, SEED + 1)


# (type, rule, box): one element, whole groups, one over, ragged
CASES = [(L.HEX27, 3, (1, 1, 1)), (L.HEX27, 3, (7, 1, 1)), (L.HEX27, 3, (2, 2, 2)), (L.HEX27, 3, (5, 3, 7)),
         (L.HEX27, 2, (3, 1, 2)), (L.HEX8, 2, (1, 1, 1)), (L.HEX8, 2, (8, 8, 1)), (L.HEX8, 2, (13, 5, 1)),
         (L.HEX8, 3, (3, 4, 5)), (L.TET4, 3, (1, 1, 1)), (L.TET4, 3, (2, 2, 2)), (L.TET4, 5, (3, 1, 1)),
         (L.TET4, 1, (3, 2, 1)), (L.TET10, 5, (1, 1, 1)), (L.TET10, 5, (3, 2, 1)), (L.TET10, 3, (2, 1, 4)),
         (L.TET10, 2, (1, 1, 3))]


@pytest.mark.parametrize("t,npts,box", CASES)
def test_matrix_free_element_kernels(ctx, t, npts, box):
    p, s, kappa = problem(ctx, t, box)
    g = L.GpuProblem.from_problem(ctx, p)
    rng = np.random.default_rng(SEED)
    u, lam = rng.standard_normal(p.n_dofs), rng.standard_normal(p.n_dofs)
    kd = L.DeviceArray(ctx, p.n_elem, data=kappa)
    ud, ld = L.DeviceArray(ctx, p.n_dofs, data=u), L.DeviceArray(ctx, p.n_dofs, data=lam)
    out, grad = L.DeviceArray(ctx, p.n_dofs), L.DeviceArray(ctx, p.n_elem)
    for f_kind in (0, 1):
        g.residual_poisson(npts, kd, f_kind, ud, out)
        assert rel(out.download(), s.residual_poisson(npts, u, kappa, f_kind)) < 1e-12, f_kind
    g.residual_poisson(npts, None, 0, ud, out)
    assert rel(out.download(), s.residual_poisson(npts, u)) < 1e-12
    g.qoi_box_derivative(npts, 0.21, 0.93, out)  # faces away from every rule's points
    assert rel(out.download(), s.qoi_box_derivative(npts, 0.21, 0.93)) < 1e-12
    g.adjoint_kappa_gradient(npts, kd, ud, ld, grad)
    free = p.constrained == 0
    Ke, _ = s.element_poisson(npts, None, 0, constrain=False)
    ue, le = (u * free)[p.elem_dofs], (lam * free)[p.elem_dofs]
    ex = -np.einsum("ei,eij,ej->e", le, Ke, ue)
    scale = np.einsum("ei,eij,ej->e", np.abs(le), np.abs(Ke), np.abs(ue)).max()
    assert np.abs(grad.download() - ex).max() <= 1e-12 * scale
    g.close()


@pytest.mark.parametrize("t,npts,box", CASES + [(L.HEX8, 2, (26, 26, 25)), (L.HEX8, 2, (33, 1, 1))])
def test_element_matrices(ctx, t, npts, box):
    """Element matrices and vectors (constrained and not, with and without
    kappa, both forcings), and the FP32 operator: each entry rounded once to
    FP32, then at most 24 of them added in FP32 (24 * 6e-8 < 2e-6)."""
    p, s, kappa = problem(ctx, t, box)
    g = L.GpuProblem.from_problem(ctx, p)
    kd = L.DeviceArray(ctx, p.n_elem, data=kappa)
    Ke, Fe = L.DeviceArray(ctx, p.n_elem * p.npe ** 2), L.DeviceArray(ctx, p.n_elem * p.npe)
    for f_kind, k, kh, con in ((0, kd, kappa, True), (1, kd, kappa, False), (1, None, None, True)):
        g.element_poisson(npts, k, f_kind, Ke, Fe, constrain=con)
        oK, oF = s.element_poisson(npts, kh, f_kind, constrain=con)
        assert rel(Ke.download(), oK.ravel()) < 1e-12, (f_kind, con)
        assert rel(Fe.download(), oF.ravel()) < 1e-12, (f_kind, con)
    b = L.DeviceArray(ctx, p.n_dofs)
    vals, rhs = s.assemble_poisson(npts, kappa, 1)
    g.assemble_poisson(npts, kd, 1, b, L.FP32)
    assert rel(g.values_fp32().astype(np.float64), vals) < 2e-6
    assert rel(b.download(), rhs) < 1e-12
    g.close()


@pytest.mark.parametrize("power", [-300, 300])
@pytest.mark.parametrize("t,npts,box", [(L.HEX27, 3, (3, 2, 1)), (L.HEX27, 2, (2, 1, 1)), (L.HEX8, 2, (3, 2, 2)),
                                        (L.HEX8, 2, (26, 26, 25)), (L.HEX8, 3, (3, 2, 2)), (L.TET4, 3, (2, 1, 1)),
                                        (L.TET10, 5, (1, 2, 1))])
def test_any_size_of_element(ctx, t, npts, box, power):
    """Coordinates times 2^power (elements of edge 1e-91 and 1e90): every product on
    the way is exact, so the results scale exactly, K and the gradient by 2^power,
    F, the residual (of u times 4^power) and the QoI derivative by 8^power."""
    p, s, kappa = problem(ctx, t, box)
    rng = np.random.default_rng(SEED + 2)
    u, lam = rng.standard_normal(p.n_dofs), rng.standard_normal(p.n_dofs)
    kd, ld = L.DeviceArray(ctx, p.n_elem, data=kappa), L.DeviceArray(ctx, p.n_dofs, data=lam)
    dpe = p.elem_dofs.shape[1]
    got = []
    for k in (0, power):
        g = L.GpuProblem(ctx, np.ldexp(p.coords, k), p.conn, p.elem_type, p.elem_dofs, p.n_dofs, p.constrained)
        ud, us = L.DeviceArray(ctx, p.n_dofs, data=u), L.DeviceArray(ctx, p.n_dofs, data=np.ldexp(u, 2 * k))
        K, F = L.DeviceArray(ctx, p.n_elem * dpe * dpe), L.DeviceArray(ctx, p.n_elem * dpe)
        R, q, grad = L.DeviceArray(ctx, p.n_dofs), L.DeviceArray(ctx, p.n_dofs), L.DeviceArray(ctx, p.n_elem)
        L.check(L.hip().lmh_element_poisson(ctx.h, g.mesh, g.dofmap, npts, kd.ptr, 0, 0, K.ptr, F.ptr))
        g.residual_poisson(npts, kd, 0, us, R)
        g.qoi_box_derivative(npts, -1e300, 1e300, q)
        g.adjoint_kappa_gradient(npts, kd, ud, ld, grad)
        got.append([np.ldexp(a.download(), -e * k) for a, e in ((K, 1), (F, 3), (R, 3), (q, 3), (grad, 1))])
        g.close()
    for name, a, b in zip(("K", "F", "residual", "qoi", "gradient"), *got):
        assert np.array_equal(a, b), name
