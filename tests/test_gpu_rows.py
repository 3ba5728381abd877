"""Assembly by rows (element forces and 3x3 blocks in buffers, gathered by
nodes and matrix rows) on meshes whose node numbers are shuffled, so that
the ranks of an element's nodes differ from element to element: the residual
against the oracle, and the MSR values and Newton's operator against the
colour-ordered assembly, whose sums have other orders (at most eight terms
an entry).  Rows too wide for the gather take the colour-ordered assembly."""
import numpy as np
import pytest

from test_gpu_split import fan

pytestmark = pytest.mark.gpu

SIMO, STVENANT = 0, 1


def shuffled(n, seed):
    from tahoe_amd import mesh as M
    m = M.cube(0, seed=seed, nxyz=n)
    p = np.random.default_rng(seed).permutation(m.nnd).astype(np.int32)   # old -> new
    X = np.empty_like(m.X)
    X[p] = m.X
    sets = {k: p[v] for k, v in m.nodesets.items()}
    return M.HexMesh(X, p[m.conn], m.mat, sets, m.shape)


def solid(m, kbc, form, model, precision):
    from tahoe_amd import api
    s = api.Solid(0)
    s.set_mesh(m.X, m.conn, m.mat)
    s.set_material(0, *api.mu_kappa(1000.0, 0.3))
    s.set_formulation(form)
    s.set_material_model(model)
    s.set_precision(precision)
    s.set_kbc(kbc.nodes, kbc.dofs, kbc.values)
    s.initialize()
    return s


def state(m):
    return 0.01 / max(m.shape or (4,)) * np.random.default_rng(8).standard_normal((m.nnd, 3)) + 0.02 * m.X


# one element; fewer and more than the 7 and 10 elements of a workgroup;
# rows past a half slice
@pytest.mark.parametrize("n", [(1, 1, 1), (3, 2, 2), (5, 3, 4), (7, 7, 7)])
@pytest.mark.parametrize("form,model,precision", [(0, SIMO, 0), (0, SIMO, 1), (0, STVENANT, 0), (0, STVENANT, 1),
                                                  (1, SIMO, 0), (1, STVENANT, 0), (1, SIMO, 1)])
def test_rows_equal_colours(n, form, model, precision):
    from oracle import oracle as O
    from tahoe_amd import api, mesh as M
    m = shuffled(n, 31)
    kbc = M.kbc_uniaxial(m, 0.01)
    kind = ((O.TL, O.TL_STVENANT), (O.Q1P0, O.Q1P0_STVENANT))[form][model]
    mu, ka = api.mu_kappa(1000.0, 0.3)
    vals, us = [], []
    for rows in (1, 0):
        s = solid(m, kbc, form, model, precision)
        s.set_tuning(api.TUNE_STIFF_ROWS, rows)
        assert s.tuning(api.TUNE_STIFF_ROWS) == rows
        u = state(m)
        s.set_displacement(u)
        R, norm = s.form_rhs()
        Ro = O.residual(kind, m.X, m.conn, m.mat, mu, ka, u, s.eqnos(), s.n_eq)
        assert np.abs(R - Ro).max() <= 1e-12 * np.abs(Ro).max()
        assert abs(norm - np.linalg.norm(Ro)) <= 1e-12 * norm
        s.form_lhs()
        s.form_lhs()          # a second pass overwrites every value
        vals.append(s.msr_values())
        x = np.random.default_rng(9).standard_normal(s.n_eq)
        b1 = s.multx(x)       # with rows, the operator written beside the MSR
        s.form_tangent()
        assert np.array_equal(s.msr_values(), vals[-1]) and np.array_equal(s.multx(x), b1)
        s.newton_correction(s.opts(lin_rtol=1e-12))
        us.append(s.displacement())
        s.close()
    tol = 1e-6 if precision and not form else 1e-13
    assert np.abs(vals[0] - vals[1]).max() <= tol * np.abs(vals[1]).max()
    assert np.abs(us[0] - us[1]).max() <= (1e-4 if precision else 1e-9) * np.abs(us[1]).max()


# 6, 7, 8 and 15 elements about a workgroup's 7; free and prescribed dofs in
# every combination, nodes with none free included
@pytest.mark.parametrize("n", [(3, 2, 1), (7, 1, 1), (2, 2, 2), (5, 3, 1)])
@pytest.mark.parametrize("precision", [0, 1])
def test_any_prescribed_dofs(n, precision):
    from tahoe_amd import api, mesh as M
    m = shuffled(n, 77)
    rng = np.random.default_rng(78)
    pick = rng.random((m.nnd, 3)) < 0.4
    pick[0] = True
    nodes, dofs = np.nonzero(pick)
    kbc = M.KBC(nodes.astype(np.int32), dofs.astype(np.int32), np.zeros(len(nodes)))
    vals, bs = [], []
    for rows in (1, 0):
        s = solid(m, kbc, 0, SIMO, precision)
        s.set_tuning(api.TUNE_STIFF_ROWS, rows)
        s.set_displacement(state(m))
        s.form_lhs()
        vals.append(s.msr_values())
        bs.append(s.multx(np.random.default_rng(9).standard_normal(s.n_eq)))
        s.close()
    tol = 1e-6 if precision else 1e-13
    assert np.abs(vals[0] - vals[1]).max() <= tol * np.abs(vals[1]).max()
    assert np.abs(bs[0] - bs[1]).max() <= 10 * tol * np.abs(bs[1]).max()


@pytest.mark.parametrize("form", [0, 1])
def test_wide_rows_take_the_colours(form):
    from oracle import oracle as O
    from tahoe_amd import api, mesh as M
    m = fan()
    kbc = M.kbc_uniaxial(m, 0.01)
    s = solid(m, kbc, form, SIMO, 0)
    try:
        assert s.tuning(api.TUNE_STIFF_ROWS) == 0
        u = state(m)
        s.set_displacement(u)
        s.form_lhs()
        mu, ka = api.mu_kappa(1000.0, 0.3)
        kind = O.Q1P0 if form else O.TL
        vo = O.stiffness(kind, m.X, m.conn, m.mat, mu, ka, u, s.eqnos(), s.n_eq, s.msr_bindx())
        assert np.abs(s.msr_values() - vo).max() <= (1e-7 if form else 1e-12) * np.abs(vo).max()
        assert s.newton(s.opts(lin_rtol=1e-12)).status == 0
    finally:
        s.close()


def test_colour_knobs_select_the_colours_and_rows_take_it_back():
    from tahoe_amd import api, mesh as M
    m = shuffled((3, 3, 3), 5)
    s = solid(m, M.kbc_uniaxial(m, 0.01), 0, SIMO, 0)
    try:
        for knob, v in ((api.TUNE_STIFF_SHAPE, 9), (api.TUNE_STIFF_CHUNK, -1), (api.TUNE_NEWTON_ASSEMBLY, 0),
                        (api.TUNE_STIFF_GATHER, 0)):
            s.set_tuning(api.TUNE_STIFF_ROWS, 1)
            assert s.tuning(api.TUNE_STIFF_ROWS) == 1
            s.set_tuning(knob, v)
            assert s.tuning(api.TUNE_STIFF_ROWS) == 0
    finally:
        s.close()


def test_tuner_times_the_assembly_by_rows():
    """tune_stiffness leaves the assembly that it reports in place, and the
    residual and the tangent are those of an untuned context."""
    from tahoe_amd import api, autotune, mesh as M
    m = M.cube(6, seed=4)
    kbc = M.kbc_uniaxial(m, 0.01)
    out = []
    for tune in (False, True):
        s = api.Solid(0)
        try:
            s.set_mesh(m.X, m.conn, m.mat)
            s.set_material(0, *api.mu_kappa(1000.0, 0.3))
            s.set_kbc(kbc.nodes, kbc.dofs, kbc.values)
            s.initialize()
            s.apply_kbc(1.0)
            if tune:
                t = autotune.tune_stiffness(s, shapes=[0], chunks=[0], reps=1)
                assert s.tuning(api.TUNE_STIFF_ROWS) == int(t["rows"])
                assert set(t["ms"]["rows"]) == {1}
            R, _ = s.form_rhs()
            s.form_lhs()
            out.append((R, s.msr_values()))
        finally:
            s.close()
    # the two assemblies sum an entry's contributions in another order
    for a, b in zip(out[0], out[1]):
        assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
