"""Formation on meshes with one long row: a ball of n surface nodes around one
hub, whose row has n + 1 blocks and 2 n - 4 incidences.  The sizes are the edges
of the flux pass (20 neighbours staged per row, places of 32 or 64 bits from
1,024 blocks on) and of the residual gather (24 records in flight per node).

Tolerance: that of test_gpu_formation.py, 1e-12 normwise against the oracle
(the same terms summed in another order)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _ball(n):
    """Hub 1 and n nodes spread over a slightly uneven unit sphere; one tet per hull triangle."""
    from scipy.spatial import ConvexHull
    k = np.arange(n) + 0.5
    z, phi = 1.0 - 2.0 * k / n, np.pi * (1.0 + 5.0 ** 0.5) * k
    r = np.sqrt(1.0 - z * z)
    p = np.stack([r * np.cos(phi), r * np.sin(phi), z], axis=1)
    hull = ConvexHull(p)
    assert len(hull.simplices) == 2 * n - 4
    x = np.vstack([[[0.03, -0.02, 0.05]], p * (1.0 + 0.05 * np.sin(5.0 * k))[:, None]])
    ien = np.hstack([np.ones((2 * n - 4, 1), int), hull.simplices + 2])
    for e in ien:
        v = x[e[:3] - 1] - x[e[3] - 1]
        if np.linalg.det(v) < 0:
            e[[2, 3]] = e[[3, 2]]
    # the hub at every local place
    for m in range(len(ien)):
        ien[m] = [ien[m], ien[m][[1, 0, 3, 2]], ien[m][[2, 3, 0, 1]], ien[m][[3, 2, 1, 0]]][m % 4]
    return np.asfortranarray(ien.astype(np.int32)), np.asfortranarray(x)


def _csr(ien, N):
    """The graph in ascending order (genadj stops at shorter rows)."""
    pairs = np.unique(np.concatenate([N * (ien[:, [a]] - 1) + ien - 1 for a in range(4)]).ravel())
    colm = np.searchsorted(pairs, N * np.arange(N + 1)) + 1
    return colm.astype(np.int32), (pairs % N + 1).astype(np.int32)


@pytest.mark.parametrize("n", [14, 15, 19, 20, 1023, 1024])
def test_formation_long_row(oracle_lib, n):
    import crimsonflowsolver_amd as cfa
    ien, x = _ball(n)
    N = n + 1
    rng = np.random.default_rng(n)
    y = np.asfortranarray(rng.normal(size=(N, 4)) * np.array([10.0, 1.0, 1.0, 1.0]))
    ac = np.asfortranarray(rng.uniform(-20, 20, size=(N, 4)))
    colm, rowp = _csr(ien, N)
    assert colm[1] - colm[0] == N
    form = cfa.ElmGMRInterior(ien, colm, rowp, N)
    got = form(y, ac, x, want_q=True)
    ref = oracle_lib.elmgmr_interior(ien, y, ac, x, colm, rowp, oracle_lib.make_params(), want_q=True)
    only = form(y, ac, x, lhs=0)[0]
    for name, a, b in zip(("res", "lhsK", "lhsP", "q", "res alone"), got + (only,), ref + (ref[0],)):
        err = float(np.abs(a - b).max() / np.abs(b).max())
        print(n, name, err, flush=True)
        assert err <= TOL, (name, err)


def test_formation_row_past_the_places(oracle_lib):
    """A hub whose row holds more than 2^20 blocks, nearly all of them touched by no
    element (zero in the result): the flux pass then counts its places among the touched
    blocks alone."""
    import crimsonflowsolver_amd as cfa
    ien, x = _ball(20)
    n, N = 21, (1 << 20) + 64
    # the hub's nodes keep their numbers, the surface's are spread over the hub's row
    num = np.concatenate([[1], 2 + np.arange(n - 1) * ((N - 2) // (n - 1))])
    ien = np.asfortranarray(num[ien - 1].astype(np.int32))
    X = np.zeros((N, 3), order="F")
    X[num - 1] = x
    rng = np.random.default_rng(20)
    y = np.asfortranarray(rng.normal(size=(N, 4)) * np.array([10.0, 1.0, 1.0, 1.0]))
    ac = np.asfortranarray(rng.uniform(-20, 20, size=(N, 4)))
    pairs = np.concatenate([np.arange(N), np.arange(N) * (N + 1)] +
                           [(N * (ien[:, [a]].astype(np.int64) - 1) + ien - 1).ravel() for a in range(4)])
    pairs = np.unique(pairs)
    colm = (np.searchsorted(pairs, N * np.arange(N + 1, dtype=np.int64)) + 1).astype(np.int32)
    rowp = (pairs % N + 1).astype(np.int32)
    assert colm[1] - colm[0] == N
    form = cfa.ElmGMRInterior(ien, colm, rowp, N)
    res, K, P, q = form(y, ac, X, want_q=True)
    rres, rK, rP, rq = oracle_lib.elmgmr_interior(ien, y, ac, X, colm, rowp, oracle_lib.make_params(), want_q=True)
    m = num - 1
    for name, a, b in (("res", res, rres), ("lhsK", K, rK), ("lhsP", P, rP), ("q", q[m], rq[m])):
        err = float(np.abs(a - b).max() / np.abs(b).max())
        print(name, err, flush=True)
        assert err <= TOL, (name, err)
