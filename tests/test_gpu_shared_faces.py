"""Many coupled faces on the same nodes: the NS solver's result against a dense
direct solve of the system with the faces' rank-one terms, on a graph whose
Schur complement is formed and on one that keeps the two passes, with fewer and with
more faces than a workgroup of the residual update keeps in LDS (256); the time
of its CG against one face's; and faces with so many shared nodes that ADDBCMUL
takes its launches per face, against one face of the same term; and a face with a
support so large that its dots take more workgroups.

Tolerance: test_gpu_schur's (1e-5 of the residual asked, condition numbers
under 1e4: 1e-2 of the solution's norm).  Without the faces' terms the solution
moves by more than 0.04.
"""
import time

import numpy as np
import pytest

from test_gpu_schur import _direct, _solve, _system

pytestmark = pytest.mark.gpu


def _faces(n, count, seed):
    rng = np.random.default_rng(seed)
    out = []
    for k in range(count):
        nodes = (3 + 2 * (k % 7) + np.arange(12)) % n
        out.append((nodes, rng.uniform(0.2, 1.0, (3, 12)), 24.0 / count))
    return out


@pytest.mark.parametrize("count", [24, 300])
@pytest.mark.parametrize("hub", [False, True], ids=["formed", "two passes"])
def test_shared_faces_against_direct(hub, count):
    import crimsonflowsolver_amd as cfa
    n = 400 if hub else 60
    edges = [(i, (i + k) % n) for i in range(n) for k in (1, 2, 3)] + ([(0, i) for i in range(1, n)] if hub else [])
    rowptr, colptr, val, A = _system(n, edges, 5)
    faces = _faces(n, count, 6)
    R = np.asfortranarray(1e4 * np.random.default_rng(7).standard_normal((4, n)))
    R[:, 30:] *= 0.1  # what the faces act on carries the right-hand side
    d, without = _direct(A, R, faces), _direct(A, R)
    assert np.linalg.norm(without - d) > 0.04 * np.linalg.norm(d)
    x = _solve(cfa, rowptr, colptr, val, R, faces)
    assert np.linalg.norm(x - d) <= 1e-2 * np.linalg.norm(d)


@pytest.mark.parametrize("kind,grid", [("CG", (48, 48, 60)), ("GMRES", (96, 96, 12))])
def test_shared_faces_cost(kind, grid):
    """100 CG iterations on a cylinder of 115,961 nodes, 30 Arnoldi steps on one of 96,525:
    with 24 coupled faces on the outlet's 1,709 and 7,041 nodes at most four times as
    long as with one."""
    import torch
    import crimsonflowsolver_amd as cfa
    from crimsonflowsolver_amd import mesh as M
    m = M.cylinder_mesh(*grid)
    colm, rowp = cfa.genadj(m.ien, m.numnp)
    y, ac = M.poiseuille_state(m, seed=5)
    ibc, _ = M.dirichlet_codes(m)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(np.asarray(a).T)).cuda()
    form = cfa.ElmGMRInterior(m.ien, colm, rowp, m.numnp, iBC=ibc, params=cfa.form_params())
    fixed, out = np.nonzero(ibc)[0], np.nonzero(m.outlet & (ibc == 0))[0]
    nabi = m.nabi()[out]
    ms = []
    for count in (1, 24):
        lhs = cfa.memLS_LHS_CREATE(m.numnp, m.numnp, rowp.size, None, colm, rowp, 1 + count)
        cfa.memLS_BC_CREATE(lhs, 1, fixed.size, 3, cfa.BC_TYPE_Dir, fixed + 1, np.zeros((3, fixed.size), order="F"))
        for k in range(count):
            cfa.memLS_BC_CREATE(lhs, 2 + k, out.size, 3, cfa.BC_TYPE_Neu, out + 1, np.asfortranarray(nabi.T))
        rhs = torch.zeros((m.numnp, 4), dtype=torch.float64, device="cuda")
        form.to_lhs(T(y), T(ac), T(m.x), rhs, lhs)
        form.bc3res(rhs, res4_layout=True)
        form.sync()
        if kind == "CG":
            ls = cfa.memLS_LS_CREATE(cfa.LS_TYPE_NS, relTol=1e-12, dimKry=1, maxItr=1, relTolIn=[0.9, 1e-30],
                                     absTolIn=[1e-30, 1e-30], maxItrIn=[1, 100])
        else:
            ls = cfa.memLS_LS_CREATE(cfa.LS_TYPE_GMRES, relTol=1e-30, absTol=1e-30, dimKry=30, maxItr=1)
        best = 1e9
        for _ in range(4):
            x = rhs.clone()
            torch.cuda.synchronize()
            t = time.perf_counter()
            cfa.memLS_SOLVE_dev(lhs, ls, 4, x, res=np.array([0.0] + [0.3 / count] * count))
            best = min(best, time.perf_counter() - t)
        assert (ls.stats("CG")["itr"] == 100) if kind == "CG" else (ls.RI["itr"] == 31)
        ms.append(1e3 * best)
    assert ms[1] <= 4.0 * ms[0], ms


def _ring(n):
    """A diagonally dominant system with D = -G^T on a ring of five blocks a row."""
    i = np.arange(n)
    cols = np.sort((i[:, None] + np.arange(-2, 3)) % n, axis=1)
    rng = np.random.default_rng(3)
    val = np.zeros((16, 5 * n), order="F")
    val[[0, 5, 10, 15]] = np.where((cols == i[:, None]).ravel(), 2.0, -0.1)
    key = {(a, b): a * 5 + k for a in range(n) for k, b in enumerate(cols[a])}
    g = 0.2 * rng.uniform(-1, 1, (3, 5 * n))
    val[[3, 7, 11]] = g
    val[12:15] = -g[:, [key[(b, a)] for a in range(n) for b in cols[a]]]
    return (5 * np.arange(n + 1) + 1).astype(np.int32), (cols.ravel() + 1).astype(np.int32), val, rng


@pytest.mark.parametrize("bits", [64, 32])
def test_face_of_many_nodes_against_direct(bits):
    """A face of 18,000 nodes (a support past 16,384, whose dots take more than four
    workgroups) and one of 100 against a sparse direct solve with the two rank-one
    terms (Woodbury).  Tolerances as above."""
    import scipy.sparse as sp
    import scipy.sparse.linalg as sla
    import torch
    import crimsonflowsolver_amd as cfa
    n = 20000
    rowptr, colptr, val, rng = _ring(n)
    faces = [(np.arange(500, 18500), 30.0), (np.arange(18400, 18500), 10.0)]
    A = sp.bsr_matrix((val.T.reshape(-1, 4, 4), colptr - 1, rowptr - 1), shape=(4 * n, 4 * n)).tocsc()
    R = 1e3 * (rng.standard_normal((n, 4)) + 1.0)
    U = np.zeros((4 * n, 2))
    lhs = cfa.memLS_LHS_CREATE(n, n, 5 * n, None, rowptr, colptr, 2)
    for f, (nodes, r) in enumerate(faces):
        v = rng.uniform(0.2, 1.0, (3, nodes.size)) / np.sqrt(nodes.size)
        for c in range(3):
            U[4 * nodes + c, f] = v[c] * np.sqrt(r)
        cfa.memLS_BC_CREATE(lhs, f + 1, nodes.size, 3, cfa.BC_TYPE_Neu, nodes + 1, np.asfortranarray(v))
    lu = sla.splu(A)
    without, Z = lu.solve(R.ravel()), lu.solve(U)
    d = without - Z @ np.linalg.solve(np.eye(2) + U.T @ Z, U.T @ without)
    lhs.set_val(4, val)
    lhs.set_precision(bits)
    ls = cfa.memLS_LS_CREATE(cfa.LS_TYPE_NS, relTol=1e-6 if bits == 64 else 1e-5, dimKry=40, maxItr=12,
                             relTolIn=[0.01, 0.01], maxItrIn=[2, 200])
    x = torch.from_numpy(R).cuda()
    cfa.memLS_SOLVE_dev(lhs, ls, 4, x, res=np.array([f[1] for f in faces]))
    assert ls.RI["suc"] == 1
    assert np.linalg.norm(without - d) > 0.1 * np.linalg.norm(d)
    assert np.linalg.norm(x.cpu().numpy().ravel() - d) <= (1e-3 if bits == 64 else 1e-2) * np.linalg.norm(d)


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("kind", ["NS", "GMRES"])
def test_large_shared_faces_against_one(kind, bits):
    """Three faces of 2,000 nodes each, all the same with a third of the coefficient,
    are one face's rank-one term.  Tolerance: both solves to 1e-6 (FP32: 1e-5) of a system
    with condition number under 1e3.  (NSSOLVER's GE takes pivots under 4.4e-16 as
    singular, and its Gram matrix holds squares of the residual: 1e-9 is out of its
    reach.)"""
    import torch
    import crimsonflowsolver_amd as cfa
    n = 6000
    rowptr, colptr, val, rng = _ring(n)
    rhs = torch.from_numpy(1e3 * (rng.standard_normal((n, 4)) + 1.0)).cuda()
    nodes = np.arange(100, 4100, 2)
    v = rng.uniform(0.2, 1.0, (3, nodes.size)) / np.sqrt(nodes.size)
    tol = 1e-6 if bits == 64 else 1e-5
    out = []
    for count in (0, 1, 3):
        lhs = cfa.memLS_LHS_CREATE(n, n, 5 * n, None, rowptr, colptr, max(count, 1))
        for f in range(count):
            cfa.memLS_BC_CREATE(lhs, f + 1, nodes.size, 3, cfa.BC_TYPE_Neu, nodes + 1, np.asfortranarray(v))
        lhs.set_val(4, val)
        lhs.set_precision(bits)
        if kind == "NS":
            ls = cfa.memLS_LS_CREATE(cfa.LS_TYPE_NS, relTol=tol, dimKry=40, maxItr=12, relTolIn=[0.01, 0.01],
                                     maxItrIn=[2, 200])
        else:
            ls = cfa.memLS_LS_CREATE(cfa.LS_TYPE_GMRES, relTol=tol, dimKry=60, maxItr=6)
        x = rhs.clone()
        cfa.memLS_SOLVE_dev(lhs, ls, 4, x, res=np.full(count, 30.0 / max(count, 1)) if count else None)
        assert ls.RI["suc"] == 1
        out.append(x.cpu().numpy())
    without, one, three = out
    assert np.linalg.norm(without - one) > 0.1 * np.linalg.norm(one)
    assert np.linalg.norm(three - one) <= (1e-3 if bits == 64 else 1e-2) * np.linalg.norm(one)
