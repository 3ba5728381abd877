"""TUNE_AMG_DEGREE: reads the degree of the fine level's smoothing (1 where
the automatic choice takes one step), and -1 gives the choice back."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 64 x 32 x 64 nodes: the first size whose fine level takes one step
@pytest.mark.parametrize("n,auto", [((8, 8, 8), 2), ((63, 31, 62), 2), ((63, 31, 63), 1)])
def test_degree_reads_what_runs_and_can_be_given_back(n, auto):
    from tahoe_amd import api, mesh as M
    m = M.cube(0, seed=8, nxyz=n)
    kbc = M.kbc_uniaxial(m, 0.002)
    s = api.Solid(0)
    try:
        s.set_mesh(m.X, m.conn, m.mat)
        s.set_material(0, *api.mu_kappa(1000.0, 0.3))
        s.set_kbc(kbc.nodes, kbc.dofs, kbc.values)
        s.set_preconditioner(api.PC_AMG)
        s.initialize()
        s.apply_kbc(1.0)
        R, _ = s.form_rhs()
        s.form_lhs()
        out = []
        for value, read in ((None, auto), (2, 2), (3, 3), (-1, auto)):
            if value is not None:
                s.set_tuning(api.TUNE_AMG_DEGREE, value)
            assert s.tuning(api.TUNE_AMG_DEGREE) == read
            x, st = s.solve(R, rtol=1e-8)
            assert st.converged
            out.append((x, st.iterations))
        assert out[3][1] == out[0][1] and np.array_equal(out[3][0], out[0][0])
        # degree 2 set by the caller is the automatic choice only where that reads 2
        assert np.array_equal(out[1][0], out[0][0]) == (auto == 2)
        assert out[2][1] < out[0][1]
        for value in (-2, 0, 1, 5):
            with pytest.raises(api.TahoeGpuError) as e:
                s.set_tuning(api.TUNE_AMG_DEGREE, value)
            assert e.value.code == 4
            assert s.tuning(api.TUNE_AMG_DEGREE) == auto
    finally:
        s.close()
