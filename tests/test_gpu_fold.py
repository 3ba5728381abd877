"""PCG's totals formed inside the kernels that need them up to 2,048 slices,
and by their own kernels beyond: on both sides of the line the direction in
the product or in its own pass gives bitwise the same correction, and the
correction is the solution."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 64 x 32 x 64 nodes (2,048 slices) and one layer of nodes more
@pytest.mark.parametrize("n", [(63, 31, 63), (63, 31, 64)])
@pytest.mark.parametrize("precision,pc", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_fused_or_not_on_both_sides(n, precision, pc):
    from tahoe_amd import api, mesh as M
    m = M.cube(0, seed=29, nxyz=n)
    kbc = M.kbc_uniaxial(m, 0.002)
    s = api.Solid(0)
    try:
        s.set_mesh(m.X, m.conn, m.mat)
        s.set_material(0, *api.mu_kappa(1000.0, 0.3))
        s.set_precision(precision)
        s.set_kbc(kbc.nodes, kbc.dofs, kbc.values)
        s.initialize()
        s.set_preconditioner(pc)
        s.apply_kbc(1.0)
        R, norm = s.form_rhs()
        s.form_lhs()
        out = []
        for fused in (-1, 0, 1):
            s.set_tuning(api.TUNE_PCG_FUSED, fused)
            x, st = s.solve(R, rtol=1e-6)
            assert st.converged
            out.append((x, st.iterations))
        for x, its in out[1:]:
            assert its == out[0][1] and np.array_equal(x, out[0][0])
        # the recurrence's residual is 1e-6 of R; the product is taken with the
        # values as assembled (FP32 in mixed precision)
        assert np.linalg.norm(R - s.multx(out[0][0])) <= (1e-4 if precision else 2e-6) * norm
    finally:
        s.close()
