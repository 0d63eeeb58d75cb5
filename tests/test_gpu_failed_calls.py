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
