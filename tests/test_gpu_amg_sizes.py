"""Multigrid-preconditioned solves at the sizes where the V-cycle's products
change form (9, 3 or 1 waves a row; lower blocks through their partners from
2^17 nodes): the solution of the Jacobi-preconditioned solve, in far fewer
iterations."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(33, 33, 34), (33, 34, 35), (45, 45, 45), (47, 47, 47), (50, 51, 51)])
def test_amg_solve_equals_jacobi(n):
    from tahoe_amd import api, mesh as M
    m = M.cube(0, seed=6, nxyz=n)
    kbc = M.kbc_uniaxial(m, 0.2 / n[2])
    s = api.Solid(0)
    try:
        s.set_mesh(m.X, m.conn, m.mat)
        s.set_material(0, *api.mu_kappa(1000.0, 0.3))
        s.set_kbc(kbc.nodes, kbc.dofs, kbc.values)
        s.initialize()
        s.apply_kbc(1.0)
        R, _ = s.form_rhs()
        s.form_lhs()
        x0, st0 = s.solve(R, rtol=1e-11)
        s.set_preconditioner(api.PC_AMG)
        x1, st1 = s.solve(R, rtol=1e-11)
        assert st0.converged and st1.converged and 4 * st1.iterations < st0.iterations
        # both residuals are below 1e-11 of R; the condition number is < 1e4 here
        assert np.abs(x1 - x0).max() <= 1e-7 * np.abs(x0).max()
    finally:
        s.close()
