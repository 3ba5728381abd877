"""batch.pack against the definition: problem by problem, each on a multiple of
64 nodes, padding nodes fully prescribed to zero, one material table.  Sizes
with and without padding, with and without predictors, materials shared and
not; and arrays that do not belong to their mesh are refused."""
import numpy as np
import pytest

from tahoe_amd import batch, mesh as M


def problem(n, seed, u0=True, nmat=1):
    m = M.cube(n, seed=seed)
    rng = np.random.default_rng(seed)
    m = M.HexMesh(m.X, m.conn, rng.integers(0, nmat, m.conn.shape[0]).astype(np.int32), m.nodesets, m.shape)
    return batch.Problem(m, M.kbc_uniaxial(m, 0.01), [1000.0 + (seed + k) % 3 for k in range(nmat)], [0.3] * nmat,
                         rng.standard_normal((m.nnd, 3)) if u0 else None)


def expected(problems):
    X, u0, conn, E, kn, kd, kv, begin = [], [], [], [], [], [], [], [0]
    for p in problems:
        a, n = begin[-1], p.mesh.nnd
        pad = (-n) % 64
        X += p.mesh.X.tolist() + [[0.0] * 3] * pad
        u0 += (p.u0.tolist() if p.u0 is not None else [[0.0] * 3] * n) + [[0.0] * 3] * pad
        conn += (p.mesh.conn + a).tolist()
        E += [p.E[k] for k in p.mesh.mat]
        kn += (np.asarray(p.kbc.nodes) + a).tolist() + [a + n + k for k in range(pad) for _ in range(3)]
        kd += list(p.kbc.dofs) + [0, 1, 2] * pad
        kv += list(p.kbc.values) + [0.0] * (3 * pad)
        begin.append(a + n + pad)
    return X, u0, conn, E, kn, kd, kv, begin


@pytest.mark.parametrize("sizes", [(3,), (2, 3, 5), (1, 7, 3, 15), (40, 3)])
@pytest.mark.parametrize("u0", ["all", "some", "none"])
def test_pack(sizes, u0):
    ps = [problem(n, 3 * i + n, u0 == "all" or (u0 == "some" and i == 0), 1 + i % 3) for i, n in enumerate(sizes)]
    pk = batch.pack(ps)
    X, U, conn, E, kn, kd, kv, begin = expected(ps)
    assert np.array_equal(pk.X, X) and np.array_equal(pk.conn, conn)
    assert (pk.u0 is None) == (u0 == "none") and (pk.u0 is None or np.array_equal(pk.u0, U))
    assert [pk.materials[m][0] for m in pk.mat] == E
    assert np.array_equal(pk.kbc.nodes, kn) and np.array_equal(pk.kbc.dofs, kd) and np.array_equal(pk.kbc.values, kv)
    assert pk.node_begin.tolist() == begin and pk.node_count.tolist() == [p.mesh.nnd for p in ps]
    assert [a.dtype for a in (pk.X, pk.conn, pk.mat, pk.kbc.nodes, pk.kbc.dofs, pk.kbc.values, pk.node_begin)] == \
        [np.float64, np.int32, np.int32, np.int32, np.int32, np.float64, np.int32]


def test_arrays_of_another_size_are_refused():
    p = problem(3, 1)
    for field, bad in (("u0", np.zeros(3)), ("u0", np.zeros((1, 3))), ("u0", p.u0[:-1])):
        q = problem(3, 1)
        setattr(q, field, bad)
        with pytest.raises(ValueError):
            batch.pack([p, q])
    q = problem(3, 1)
    q.mesh = M.HexMesh(q.mesh.X, q.mesh.conn, q.mesh.mat[:1], q.mesh.nodesets, q.mesh.shape)
    with pytest.raises(ValueError):
        batch.pack([p, q])


def test_no_problems_are_refused():
    with pytest.raises(ValueError):
        batch.pack([])
