"""A call that ends in an error after it launched its kernels leaves nothing
behind that the next call would see."""
import pytest

import libmesh_amd as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [L.FP64, L.FP32])
def test_degenerate_flag_of_a_failed_call(ctx, precision):
    """An assembly refused for its scatter mode after the element kernel went out,
    on a mesh whose last element is degenerate; then at once a valid mesh."""
    p = L.Problem(24, L.HEX27)
    xyz = p.coords.copy()
    xyz[p.conn[-1, 26], 0] += 1.5 / 24  # the centre node through its +x face
    bad = L.GpuProblem(ctx, xyz, p.conn, p.elem_type, p.elem_dofs, p.n_dofs, p.constrained)
    q = L.Problem(2, L.HEX8)
    good = L.GpuProblem.from_problem(ctx, q)
    b, c = L.DeviceArray(ctx, p.n_dofs), L.DeviceArray(ctx, q.n_dofs)
    good.assemble_poisson(2, None, 0, c, precision)
    for _ in range(5):
        with pytest.raises(L.LmhError, match="unknown scatter mode"):
            bad.assemble_poisson(3, None, 0, b, precision, 99)
        good.assemble_poisson(2, None, 0, c, precision)
    with pytest.raises(L.LmhError, match="degenerate"):
        bad.assemble_poisson(3, None, 0, b, precision)
    good.assemble_poisson(2, None, 0, c, precision)
    bad.close()
    good.close()


@pytest.mark.parametrize("t,npts,box", [(L.HEX8, 2, (2, 2, 2)), (L.HEX8, 2, (26, 26, 25)), (L.HEX8, 3, (2, 2, 2)),
                                        (L.HEX27, 3, (2, 2, 2)), (L.HEX27, 2, (2, 2, 2)), (L.TET4, 3, (2, 2, 2)),
                                        (L.TET10, 5, (2, 2, 2))])
def test_nan_coordinate_is_refused(ctx, t, npts, box):
    """By every element kernel alike: a determinant that is not a number is not positive"""
    p = L.Problem(box[0], t, 1, L.ALL_FACES, box[1], box[2])
    xyz = p.coords.copy()
    xyz[p.conn[p.n_elem // 2, 0], 1] = float("nan")
    g = L.GpuProblem(ctx, xyz, p.conn, p.elem_type, p.elem_dofs, p.n_dofs, p.constrained)
    b, u = L.DeviceArray(ctx, p.n_dofs), L.DeviceArray(ctx, p.n_dofs)
    k, grad = L.DeviceArray(ctx, p.n_elem), L.DeviceArray(ctx, p.n_elem)
    u.zero()
    k.zero()
    for call in (lambda: g.assemble_poisson(npts, None, 0, b), lambda: g.assemble_poisson(npts, None, 1, b, L.FP32),
                 lambda: g.residual_poisson(npts, None, 0, u, b), lambda: g.qoi_box_derivative(npts, 0.0, 1.0, b),
                 lambda: g.adjoint_kappa_gradient(npts, k, u, u, grad)):
        with pytest.raises(L.LmhError, match="degenerate"):
            call()
    g.close()
