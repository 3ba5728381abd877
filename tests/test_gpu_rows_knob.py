"""TUNE_STIFF_ROWS = 1 after TUNE_NEWTON_ASSEMBLY = 1: Newton's tangent is
assembled by rows again, bitwise as in a context that was never tuned, and
the tuner's report of the assembly in use is the one Newton takes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def solid(precision=0):
    from tahoe_amd import api, mesh as M
    m = M.cube(5, seed=4)
    kbc = M.kbc_uniaxial(m, 0.01)
    s = api.Solid(0)
    s.set_mesh(m.X, m.conn, m.mat)
    s.set_material(0, *api.mu_kappa(1000.0, 0.3))
    s.set_precision(precision)
    s.set_kbc(kbc.nodes, kbc.dofs, kbc.values)
    s.initialize()
    s.apply_kbc(1.0)
    return s


def tangent(s):
    """MSR values after Newton's tangent (only the assemblies through the MSR
    write them) and one correction's displacement."""
    s.form_tangent()
    v = s.msr_values()
    s.newton_correction(s.opts(lin_rtol=1e-10))
    u = s.displacement()
    s.reset_step()
    s.apply_kbc(1.0)
    return v, u


@pytest.mark.parametrize("precision", [0, 1])
def test_rows_taken_back_after_the_operator_path(precision):
    from tahoe_amd import api
    a, b = solid(precision), solid(precision)
    try:
        b.set_tuning(api.TUNE_NEWTON_ASSEMBLY, 1)
        assert b.tuning(api.TUNE_STIFF_ROWS) == 0
        b.newton_correction(b.opts(lin_rtol=1e-10))
        b.reset_step()
        b.apply_kbc(1.0)
        b.set_tuning(api.TUNE_STIFF_ROWS, 1)
        assert b.tuning(api.TUNE_STIFF_ROWS) == 1
        for x, y in zip(tangent(a), tangent(b)):
            assert np.array_equal(x, y)
        # the knob off again: the operator path that was set before
        b.set_tuning(api.TUNE_STIFF_ROWS, 0)
        before = b.msr_values()
        b.set_displacement(b.displacement() * 1.5)
        b.form_tangent()
        assert np.array_equal(b.msr_values(), before)
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("rows_ms,rows", [(0.5, True), (2.0, False)])
def test_tuner_reports_the_assembly_newton_takes(monkeypatch, rows_ms, rows):
    """With times given by the test: the operator path is the best
    colour-ordered form, and the rows are faster or slower than it."""
    from tahoe_amd import api, autotune

    def timed(solid, reps, run_correction=None):
        if solid.tuning(api.TUNE_STIFF_ROWS) == 1:
            return rows_ms
        return 1.0 if solid.tuning(api.TUNE_NEWTON_ASSEMBLY) == 1 else 1.5

    monkeypatch.setattr(autotune, "_time_stiffness", timed)
    a, b = solid(), solid()
    try:
        t = autotune.tune_stiffness(b, shapes=[0], chunks=[0], reps=1, run_correction=lambda: None)
        assert t["rows"] is rows and t["assembly"] == 1
        assert b.tuning(api.TUNE_STIFF_ROWS) == int(rows)
        va, _ = tangent(a)
        b.form_lhs()
        b.set_displacement(1.5 * b.displacement())
        before = b.msr_values()
        b.form_tangent()
        # the assembly by rows writes the MSR values, the operator path does not
        assert np.array_equal(b.msr_values(), before) is not rows
        b.reset_step()
        b.apply_kbc(1.0)
        if rows:
            assert np.array_equal(tangent(b)[0], va)
    finally:
        a.close()
        b.close()
