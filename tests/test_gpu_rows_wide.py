"""The widest rows that the assembly by rows takes: axis nodes of 12 elements
and 26 upper blocks (a hexahedral grid has 8 and 14), so that a row's eight
lanes zero, add and read each other's sums many times over.  Against the
oracle, twice in a row bitwise, and after a pass at another state."""
import numpy as np
import pytest

from test_gpu_split import fan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form,precision", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_rows_of_many_elements(form, precision):
    from oracle import oracle as O
    from tahoe_amd import api, mesh as M
    m = fan(nq=6, nz=40)
    kbc = M.kbc_uniaxial(m, 0.01)
    mu, ka = api.mu_kappa(1000.0, 0.3)
    rng = np.random.default_rng(8)
    u = 0.002 * rng.standard_normal((m.nnd, 3)) + 0.02 * m.X
    s = api.Solid(0)
    try:
        s.set_mesh(m.X, m.conn, m.mat)
        s.set_material(0, mu, ka)
        s.set_formulation(form)
        s.set_precision(precision)
        s.set_kbc(kbc.nodes, kbc.dofs, kbc.values)
        s.initialize()
        assert s.tuning(api.TUNE_STIFF_ROWS) == 1
        kind = O.Q1P0 if form else O.TL
        x = rng.standard_normal(s.n_eq)
        out = []
        for state in (-0.5 * u, u, u):
            s.set_displacement(state)
            R, _ = s.form_rhs()
            s.form_lhs()
            out.append((R, s.msr_values(), s.multx(x)))
        for a, b in zip(out[1], out[2]):
            assert np.array_equal(a, b)
        R, v, y = out[2]
        b = s.msr_bindx()
        Ro = O.residual(kind, m.X, m.conn, m.mat, mu, ka, u, s.eqnos(), s.n_eq)
        vo = O.stiffness(kind, m.X, m.conn, m.mat, mu, ka, u, s.eqnos(), s.n_eq, b)
        assert np.abs(R - Ro).max() <= 1e-12 * np.abs(Ro).max()
        # the Q1P0 tangent is a forward difference with step 1e-7
        assert np.abs(v - vo).max() <= (1e-7 if form else 1e-6 if precision else 1e-12) * np.abs(vo).max()
        # the product uses the values as they are, in the operator's precision
        yo = O.msr_multx(b, v, x)
        assert np.abs(y - yo).max() <= (1e-6 if precision else 1e-12) * np.abs(yo).max()
    finally:
        s.close()
