"""The Schur complement formed for the NS solver's CG (crimson_ls_solve*)
where its pattern and rows can go wrong: graphs whose two-ring is the whole
graph, rows at and past the 16-lane and 80-entry turns, a column offset past
2 bytes, a hub node whose row is too long to be formed (the two-pass
operator), and two coupled faces that share nodes.  Reference: a dense direct
solve of the scaled system.  Tolerance: the NS solver is asked for 1e-5 of the
residual norm; the scaled systems here have condition numbers under 1e4
(asserted), so the solution is within 1e-1 of its norm at worst; 1e-2 is asked.  A
dropped face moves it by more than 0.04.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(n, edges, seed):
    """A diagonally dominant 4x4-block system on the graph `edges` with D =
    -G^T blockwise, as the NS solver's structure asks (K near the identity, L
    symmetric positive): (rowptr, colptr 1-based, Val(16, nnz), dense)."""
    rng = np.random.default_rng(seed)
    adj = [set([i]) for i in range(n)]
    for a, b in edges:
        adj[a].add(b)
        adj[b].add(a)
    cols = [sorted(s) for s in adj]
    rp = np.concatenate([[0], np.cumsum([len(c) for c in cols])])
    deg = np.array([len(c) for c in cols], float)
    A = np.zeros((4 * n, 4 * n))
    for i in range(n):
        for j in cols[i]:
            s = 1.0 / np.sqrt(deg[i] * deg[j])
            if i == j:
                A[4 * i:4 * i + 3, 4 * i:4 * i + 3] = np.eye(3) * 2.0 + 0.1 * rng.uniform(-1, 1, (3, 3))
                A[4 * i + 3, 4 * i + 3] = 1.0 + rng.uniform()
            else:
                A[4 * i:4 * i + 3, 4 * j:4 * j + 3] = 0.3 * s * rng.uniform(-1, 1, (3, 3))
            if i <= j:
                g = 0.4 * s * rng.uniform(-1, 1, 3)
                A[4 * i:4 * i + 3, 4 * j + 3] = g
                A[4 * j + 3, 4 * i:4 * i + 3] = -g
                h = 0.4 * s * rng.uniform(-1, 1, 3) if i != j else g
                A[4 * j:4 * j + 3, 4 * i + 3] = h
                A[4 * i + 3, 4 * j:4 * j + 3] = -h
                if i != j:
                    A[4 * i + 3, 4 * j + 3] = A[4 * j + 3, 4 * i + 3] = -0.4 * s * rng.uniform()
    val = np.zeros((16, int(rp[-1])), order="F")
    for i in range(n):
        for k, j in enumerate(cols[i]):
            val[:, rp[i] + k] = A[4 * i:4 * i + 4, 4 * j:4 * j + 4].ravel()
    return rp.astype(np.int32) + 1, np.concatenate(cols).astype(np.int32) + 1, val, A


def _solve(cfa, rowptr, colptr, val, R, faces=()):
    n = rowptr.size - 1
    lhs = cfa.memLS_LHS_CREATE(n, n, colptr.size, None, rowptr, colptr, len(faces))
    for f, (nodes, v, _) in enumerate(faces):
        cfa.memLS_BC_CREATE(lhs, f + 1, nodes.size, 3, cfa.BC_TYPE_Neu, nodes + 1, np.asfortranarray(v))
    ls = cfa.memLS_LS_CREATE(cfa.LS_TYPE_NS, relTol=1e-5, dimKry=40, maxItr=20, relTolIn=[0.1, 0.1],
                             maxItrIn=[5, 400])
    out = []
    for _ in range(2):  # the second solve reuses the handle's pattern
        x = R.copy(order="F")
        cfa.memLS_SOLVE(lhs, ls, 4, x, val, res=np.array([f[2] for f in faces]) if faces else None)
        out.append(x)
    assert np.array_equal(out[0], out[1])
    assert ls.RI["suc"] == 1
    return out[0]


def _direct(A, R, faces=()):
    n = R.shape[1]
    B = A.copy()
    for nodes, v, r in faces:
        u = np.zeros(4 * n)
        for c in range(3):
            u[4 * nodes + c] = v[c]
        B += r * np.outer(u, u)
    d = 1.0 / np.sqrt(np.abs(np.diag(A)))
    assert np.linalg.cond(d[:, None] * B * d[None, :]) < 1e4
    return np.linalg.solve(B, R.T.ravel()).reshape(n, 4).T


def _graphs():
    ring = lambda n, w: [(i, (i + k) % n) for i in range(n) for k in range(1, w + 1)]  # noqa: E731
    yield "one row tile and one more", 17, ring(17, 1)
    yield "two-ring rows of 81", 200, ring(200, 20)
    yield "two-ring is the whole graph", 90, ring(90, 23)
    yield "hub: a row too long to be formed", 700, [(0, i) for i in range(1, 700)] + ring(700, 1)


@pytest.mark.parametrize("name,n,edges", list(_graphs()), ids=[g[0] for g in _graphs()])
def test_schur_graphs(name, n, edges):
    import crimsonflowsolver_amd as cfa
    rowptr, colptr, val, A = _system(n, edges, 3)
    R = np.asfortranarray(1e4 * np.random.default_rng(4).standard_normal((4, n)))
    x, d = _solve(cfa, rowptr, colptr, val, R), _direct(A, R)
    assert np.linalg.norm(x - d) <= 1e-2 * np.linalg.norm(d), name


def test_schur_far_columns():
    """A chain with links over 40,000 numbers: 4-byte columns."""
    import crimsonflowsolver_amd as cfa
    import scipy.sparse as sp
    import scipy.sparse.linalg as sla
    n = 40100
    i = np.arange(n)
    pairs = np.concatenate([np.stack([i[:-1], i[1:]], 1), [[0, n - 1], [5, 40050]]])
    a = np.concatenate([i, pairs[:, 0], pairs[:, 1]])
    b = np.concatenate([i, pairs[:, 1], pairs[:, 0]])
    o = np.lexsort((b, a))
    a, b = a[o], b[o]
    rng = np.random.default_rng(7)
    val = np.zeros((16, a.size), order="F")
    key = {(p, q): k for k, (p, q) in enumerate(zip(a, b))}
    for k, (p, q) in enumerate(zip(a, b)):
        if p == q:
            val[[0, 5, 10], k] = 2.0
            val[15, k] = 2.0
        elif p < q:
            t = key[(q, p)]
            for kk, tt in ((k, t), (t, k)):
                g = 0.3 * rng.uniform(-1, 1, 3)
                val[[3, 7, 11], kk] = g
                val[[12, 13, 14], tt] = -g
            val[15, k] = val[15, t] = -0.3
    rowptr = (np.searchsorted(a, np.arange(n + 1)) + 1).astype(np.int32)
    R = np.asfortranarray(1e4 * rng.standard_normal((4, n)))
    x = _solve(cfa, rowptr, (b + 1).astype(np.int32), val, R)
    A = sp.bsr_matrix((val.T.reshape(-1, 4, 4), b, rowptr - 1), shape=(4 * n, 4 * n)).tocsc()
    d = sla.spsolve(A, R.T.ravel()).reshape(n, 4).T
    assert np.linalg.norm(x - d) <= 1e-2 * np.linalg.norm(d)


def test_schur_faces_sharing_nodes():
    import crimsonflowsolver_amd as cfa
    n = 60
    rowptr, colptr, val, A = _system(n, [(i, (i + k) % n) for i in range(n) for k in (1, 2, 3)], 5)
    rng = np.random.default_rng(6)
    faces = [(np.arange(4, 14), rng.uniform(0.2, 1.0, (3, 10)), 7.0),
             (np.arange(10, 25), rng.uniform(0.2, 1.0, (3, 15)), 4.0)]
    R = np.asfortranarray(1e4 * rng.standard_normal((4, n)))
    x, d, without = _solve(cfa, rowptr, colptr, val, R, faces), _direct(A, R, faces), _direct(A, R)
    assert np.linalg.norm(without - d) > 0.04 * np.linalg.norm(d)
    assert np.linalg.norm(x - d) <= 1e-2 * np.linalg.norm(d)
