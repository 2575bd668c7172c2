"""The NS solver's CG in two launches per iteration (up to 65,536 rows) against three:
a cylinder of 34,272 nodes, and the same cylinder twice in one matrix (68,544 rows,
an outlet face each).  Every dot product of the doubled solve is twice the single
one's, so that the iterations agree up to rounding, and both copies' solutions with
the single one.

Tolerance: 1e-8 normwise (rounding of 1e-16 grown over some hundred iterations; a
wrong direction, face term or state shows at the inner tolerances, 1e-2)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-8


@pytest.mark.parametrize("precision", [64, 32])
def test_two_launches_against_three(precision):
    import torch
    import crimsonflowsolver_amd as cfa
    from crimsonflowsolver_amd import mesh as M
    from crimsonflowsolver_amd.timestep import ns_solver
    m = M.cylinder_mesh(20, 20, 95)
    y, ac = M.poiseuille_state(m, seed=5)
    n = m.numnp
    ibc, _ = M.dirichlet_codes(m)
    fixed, out = np.nonzero(ibc)[0], np.nonzero(m.outlet & (ibc == 0))[0]
    nabi = m.nabi()[out]
    par = cfa.form_params(precision=precision)
    got, its = [], []
    for copies in (1, 2):
        N = copies * n
        assert (N > 1 << 16) == (copies == 2)
        rep = lambda a: np.asfortranarray(np.concatenate([a] * copies))
        ien = np.asfortranarray(np.concatenate([m.ien + k * n for k in range(copies)]).astype(np.int32))
        colm, rowp = cfa.genadj(ien, N)
        form = cfa.ElmGMRInterior(ien, colm, rowp, N, iBC=rep(ibc).astype(np.int32), params=par)
        lhs = cfa.memLS_LHS_CREATE(N, N, rowp.size, None, colm, rowp, 1 + copies)
        fx = np.concatenate([fixed + k * n for k in range(copies)])
        cfa.memLS_BC_CREATE(lhs, 1, fx.size, 3, cfa.BC_TYPE_Dir, fx + 1, np.zeros((3, fx.size), order="F"))
        for k in range(copies):
            cfa.memLS_BC_CREATE(lhs, 2 + k, out.size, 3, cfa.BC_TYPE_Neu, out + k * n + 1, np.asfortranarray(nabi.T))
        T = lambda a: torch.from_numpy(np.ascontiguousarray(np.asarray(a).T)).cuda()
        res4 = torch.zeros((N, 4), dtype=torch.float64, device="cuda")
        form.to_lhs(T(rep(y)), T(rep(ac)), T(rep(m.x)), res4, lhs)
        form.bc3res(res4, res4_layout=True)
        form.sync()
        res4 /= res4[:n].norm()
        ls = ns_solver(maxItr=4)
        cfa.memLS_SOLVE_dev(lhs, ls, 4, res4, res=np.array([0.0] + [0.5] * copies))
        got.append(res4.cpu().numpy().reshape(copies, n, 4))
        its.append([ls.stats(k)["itr"] for k in ("RI", "GM", "CG")])
    one, two = got[0][0], got[1]
    errs = [float(np.abs(t - one).max() / np.abs(one).max()) for t in two]
    print(precision, its, errs)
    assert its[0] == its[1]
    assert max(errs) <= (TOL if precision == 64 else 1e-3)
