"""PCG with a slice's rows shared by several waves (the untuned choice up to
98,304 nodes): bitwise the iterates of one lane per row with the direction
in its own pass, on both sides of every size at which the number of waves
changes, for rows wider than one round of the workgroup, and for a batch
whose segments end inside a group of four slices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def fan(nq=12, nz=3, seed=3):
    """Quadrilaterals (centre, rim, corner, rim) around an axis, extruded:
    the axis nodes belong to 2 nq elements and have 3 (2 nq + 1) neighbours."""
    from tahoe_amd import mesh as M
    rng = np.random.default_rng(seed)
    t = np.pi * np.arange(2 * nq) / nq
    r = np.where(np.arange(2 * nq) % 2 == 0, 1.0, 1.3)
    plane = np.concatenate([[[0.0, 0.0]], np.stack([r * np.cos(t), r * np.sin(t)], 1)])
    m = len(plane)
    X = np.concatenate([np.column_stack([plane, np.full(m, 0.4 * k)]) for k in range(nz + 1)])
    X += 0.01 * rng.standard_normal(X.shape)
    q = np.array([[0, 1 + 2 * i, 2 + 2 * i, 1 + (2 * i + 2) % (2 * nq)] for i in range(nq)])
    conn = np.concatenate([np.concatenate([q + k * m, q + (k + 1) * m], 1) for k in range(nz)])
    sets = {1: np.arange(m, dtype=np.int32), 2: np.arange(nz * m, (nz + 1) * m, dtype=np.int32)}
    return M.HexMesh(X, conn.astype(np.int32), np.zeros(len(conn), np.int32), sets, None)


def corrections(s, pc, lin_maxit):
    from tahoe_amd import api
    out = []
    s.set_preconditioner(pc)
    for fused, variant in ((-1, -1), (0, 2), (0, 0)):
        s.set_tuning(api.TUNE_PCG_FUSED, fused)
        s.set_tuning(api.TUNE_SPMV_XCD, variant)
        s.set_tuning(api.TUNE_PCG_PERSIST, 0)
        s.reset_step()
        s.apply_kbc(1.0)
        st = s.newton_correction(s.opts(lin_rtol=1e-9, lin_maxit=lin_maxit))
        out.append((s.displacement(), st.lin_iterations))
    for u, its in out[1:]:
        assert its == out[0][1]
        assert np.array_equal(u, out[0][0])
    assert np.abs(out[0][0]).max() > 0 and np.isfinite(out[0][0]).all()


def solid(m, kbc, precision):
    from tahoe_amd import api
    s = api.Solid(0)
    s.set_mesh(m.X, m.conn, m.mat)
    s.set_material(0, *api.mu_kappa(1000.0, 0.3))
    s.set_precision(precision)
    s.set_kbc(kbc.nodes, kbc.dofs, kbc.values)
    s.initialize()
    return s


# element counts whose node counts are 64 x 256 and 64 x 640 (the last sizes
# of 9 and of 5 waves), one row of nodes more, and past 98,304 nodes
@pytest.mark.parametrize("n", [(1, 1, 1), (31, 15, 31), (31, 16, 31), (31, 31, 39), (31, 32, 39), (47, 47, 42)])
@pytest.mark.parametrize("precision,pc", [(0, 0), (1, 1)])
def test_split_rows_bitwise(n, precision, pc):
    from tahoe_amd import mesh as M
    m = M.cube(0, seed=17, nxyz=n)
    s = solid(m, M.kbc_uniaxial(m, 0.3 / n[2] / 10), precision)
    try:
        corrections(s, pc, 37)
    finally:
        s.close()


@pytest.mark.parametrize("precision,pc", [(0, 1), (1, 0)])
def test_split_rows_wider_than_a_round(precision, pc):
    from tahoe_amd import mesh as M
    m = fan()
    s = solid(m, M.kbc_uniaxial(m, 0.01), precision)
    try:
        corrections(s, pc, 200)
    finally:
        s.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_split_rows_batch_bitwise(precision):
    from tahoe_amd import api, batch, rve
    # 1, 2, 6, 16 and 35 slices: groups of four end short in most segments
    probs = [rve.Request(i, L, api.TOTAL_LAGRANGIAN, 0.3, 40 + i).problem() for i, L in enumerate([2, 4, 6, 9, 12])]
    pk = batch.pack(probs)
    res = []
    for fused, variant in ((-1, -1), (0, 2), (1, 5)):
        s = batch.make_solid(pk, precision=precision)
        try:
            s.set_tuning(api.TUNE_PCG_PERSIST, 0)
            s.set_tuning(api.TUNE_PCG_FUSED, fused)
            s.set_tuning(api.TUNE_SPMV_XCD, variant)
            us, st = batch.solve_one_step_partial(s, pk, api.Solid.opts(lin_rtol=1e-8))
            res.append((us, [(x.status, x.iterations, x.lin_iterations) for x in st]))
        finally:
            s.close()
    for us, st in res[1:]:
        assert st == res[0][1]
        assert all(np.array_equal(a, b) for a, b in zip(us, res[0][0]))
    assert all(x[0] == 0 for x in res[0][1])


# the first size whose rows three waves share again (2^17 nodes: FP32 by plain
# loads, FP64 by non-temporal ones) and the node row before it, the first size
# that takes the slices in index order (2^19), and rows of 75 blocks, more than
# a round of the three waves
@pytest.mark.parametrize("n", [(63, 31, 63), (63, 31, 62), (127, 63, 63), None])
@pytest.mark.parametrize("precision,pc", [(0, 0), (1, 1)])
def test_shared_rows_bitwise(n, precision, pc):
    from tahoe_amd import mesh as M
    m = fan(nz=5300) if n is None else M.cube(0, seed=23, nxyz=n)
    s = solid(m, M.kbc_uniaxial(m, 0.001), precision)
    try:
        corrections(s, pc, 21)
    finally:
        s.close()


def test_streamed_batch_bitwise():
    """A batch whose operator exceeds the last-level cache (40 cubes of 18^3:
    296 MB in FP32) by non-temporal loads, and by plain ones."""
    from tahoe_amd import api, batch, rve
    pk = batch.pack([rve.Request(i, 18, api.TOTAL_LAGRANGIAN, 0.3, 90 + i).problem() for i in range(40)])
    res = []
    for variant in (-1, 2):
        s = batch.make_solid(pk, precision=api.MIXED)
        try:
            s.set_tuning(api.TUNE_SPMV_XCD, variant)
            us, st = batch.solve_one_step_partial(s, pk, api.Solid.opts(lin_rtol=1e-3))
            res.append((us, [(x.status, x.iterations, x.lin_iterations) for x in st]))
        finally:
            s.close()
    assert res[0][1] == res[1][1] and all(x[0] == 0 for x in res[0][1])
    assert all(np.array_equal(a, b) for a, b in zip(res[0][0], res[1][0]))
