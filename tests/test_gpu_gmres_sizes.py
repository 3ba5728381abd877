"""GMRES at the sizes where its product changes form (nine waves share a row
up to 40,960 nodes, three beyond) and on rows wider than a round of either:
one correction against a tight PCG correction of the same system."""
import numpy as np
import pytest

from test_gpu_split import fan

pytestmark = pytest.mark.gpu


# 32 x 32 x 40 = 40,960 nodes, one layer of nodes more, rows of 75 blocks on
# either side of the line
@pytest.mark.parametrize("n", [(31, 31, 39), (31, 31, 40), "fan", "long fan"])
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("pc", [0, 1])
def test_gmres_equals_pcg(n, precision, pc):
    from tahoe_amd import api, mesh as M
    m = fan() if n == "fan" else fan(nz=1700) if n == "long fan" else M.cube(0, seed=37, nxyz=n)
    if n == "long fan":
        # every eighth layer fixed, so that the system stays well conditioned
        fixed = np.nonzero((np.arange(m.nnd) // 25) % 8 == 0)[0].astype(np.int32)
        z = np.zeros(3 * len(fixed))
        kbc = M.KBC(np.repeat(fixed, 3), np.tile(np.arange(3, dtype=np.int32), len(fixed)), z)
    else:
        kbc = M.kbc_uniaxial(m, 0.002)
    s = api.Solid(0)
    try:
        s.set_mesh(m.X, m.conn, m.mat)
        s.set_material(0, *api.mu_kappa(1000.0, 0.3))
        s.set_precision(precision)
        s.set_kbc(kbc.nodes, kbc.dofs, kbc.values)
        s.initialize()
        s.set_preconditioner(pc)
        u = 0.001 * np.random.default_rng(3).standard_normal((m.nnd, 3)) / max(m.shape or (4,))
        s.set_displacement(u)
        s.apply_kbc(1.0)
        R, _ = s.form_rhs()
        s.form_lhs()
        x0, st0 = s.solve(R, rtol=1e-10)
        # one cycle: the tolerance is relative to the residual at its start
        s.set_linear_solver(api.LIN_GMRES, 600)
        x1, st1 = s.solve(R, rtol=1e-9, maxit=20000)
        assert st0.converged and st1.converged and st1.iterations > 5
        # condition numbers below 1e5: two digits of margin above 1e-9 x 1e5
        assert np.abs(x1 - x0).max() <= 1e-3 * np.abs(x0).max()
        y = s.multx(x1)
        # residual in the values' precision (FP32 in mixed precision)
        assert np.linalg.norm(R - y) <= (1e-4 if precision else 1e-7) * np.linalg.norm(R)
    finally:
        s.close()
