"""A node that no element uses keeps its free dofs as empty rows: zero MSR
diagonal and values, 1/diag zero.  On a context that held a larger mesh
before, so that its buffers carry that mesh's values, both assemblies give
the same zeros, and a product before a solve does not change the solve."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def with_isolated(m, at):
    """m with one more node, number `at`, that no element uses."""
    from tahoe_amd import mesh as M
    X = np.insert(m.X, at, [[5.0, 5.0, 5.0]], axis=0)
    up = lambda a: (a + (a >= at)).astype(np.int32)  # noqa: E731
    return M.HexMesh(X, up(m.conn), m.mat, {k: up(v) for k, v in m.nodesets.items()}, m.shape)


def set_up(s, m, kbc, form, precision):
    from tahoe_amd import api
    s.set_mesh(m.X, m.conn, m.mat)
    s.set_material(0, *api.mu_kappa(1000.0, 0.3))
    s.set_formulation(form)
    s.set_precision(precision)
    s.set_kbc(kbc.nodes, kbc.dofs, kbc.values)
    s.initialize()


# the node first, inside a slice and last
@pytest.mark.parametrize("at", [0, 70, 125])
@pytest.mark.parametrize("form,precision", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_isolated_node_has_empty_rows(at, form, precision):
    from tahoe_amd import api, mesh as M
    big, m = M.cube(8, seed=2), with_isolated(M.cube(4, seed=3), at)
    kbc = M.kbc_uniaxial(m, 0.01)
    vals, xs = [], []
    for rows in (1, 0):
        s = api.Solid(0)
        try:
            s.set_tuning(api.TUNE_STIFF_ROWS, rows)
            set_up(s, big, M.kbc_uniaxial(big, 0.01), form, precision)
            s.form_lhs()
            assert np.abs(s.msr_values()[:s.n_eq]).min() > 0
            set_up(s, m, kbc, form, precision)
            assert s.tuning(api.TUNE_STIFF_ROWS) == rows
            s.apply_kbc(1.0)
            R, _ = s.form_rhs()
            eq = s.eqnos()[at] - 1
            assert (eq >= 0).all() and np.all(R[eq] == 0.0)
            s.form_lhs()
            v = s.msr_values()
            assert np.all(v[eq] == 0.0) and np.array_equal(s.copy_diagonal(), v[:s.n_eq])
            b = s.msr_bindx()
            assert all(b[e] == b[e + 1] for e in eq)        # no off-diagonal entries
            x0, st0 = s.solve(R, rtol=1e-10)
            y = s.multx(np.ones(s.n_eq))
            assert np.all(y[eq] == 0.0) and np.isfinite(y).all()
            x1, st1 = s.solve(R, rtol=1e-10)
            assert st0.converged and st1.iterations == st0.iterations and np.array_equal(x0, x1)
            assert np.all(x1[eq] == 0.0)
            vals.append(v)
            xs.append(x1)
        finally:
            s.close()
    # sums of at most eight terms in another order, in the assembly's precision
    tol = 1e-6 if precision and not form else 1e-13
    assert np.abs(vals[0] - vals[1]).max() <= tol * np.abs(vals[1]).max()
    assert np.abs(xs[0] - xs[1]).max() <= (1e-4 if precision else 1e-8) * np.abs(xs[1]).max()
