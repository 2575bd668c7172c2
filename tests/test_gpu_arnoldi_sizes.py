"""GMRES over the sizes at which its Arnoldi step changes its launches and its split
(65,536, 131,072 and 262,144 entries): a cylinder of 14,933 nodes once, twice, four
and eight times in one matrix (59,732 to 477,856 entries).  Every dot product of the
copies' solve is a multiple of the single one's, so that the iterations agree up to
rounding, and every copy's solution with the single one's.

Tolerance: 1e-8 normwise (rounding of 1e-16, grown over 45 steps of a
reorthogonalised basis; a wrong coefficient or a wrong last step shows at the
reduction reached, 1e-3 and above)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-8


@pytest.mark.parametrize("sD", [1, 15, 17])
def test_gmres_sizes_agree(sD):
    import torch
    import crimsonflowsolver_amd as cfa
    from crimsonflowsolver_amd import mesh as M
    m = M.cylinder_mesh(12, 12, 108)
    y, ac = M.poiseuille_state(m, seed=5)
    n = m.numnp
    ibc, _ = M.dirichlet_codes(m)
    fixed, out = np.nonzero(ibc)[0], np.nonzero(m.outlet & (ibc == 0))[0]
    nabi = m.nabi()[out]
    ref = None
    for copies in (1, 2, 4, 8):
        N = copies * n
        rep = lambda a: np.asfortranarray(np.concatenate([a] * copies))
        ien = np.asfortranarray(np.concatenate([m.ien + k * n for k in range(copies)]).astype(np.int32))
        colm, rowp = cfa.genadj(ien, N)
        form = cfa.ElmGMRInterior(ien, colm, rowp, N, iBC=rep(ibc).astype(np.int32))
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
        ls = cfa.memLS_LS_CREATE(cfa.LS_TYPE_GMRES, relTol=1e-9, dimKry=sD, maxItr=3)
        cfa.memLS_SOLVE_dev(lhs, ls, 4, res4, res=np.array([0.0] + [0.5] * copies))
        x, st = res4.cpu().numpy().reshape(copies, n, 4), ls.stats("RI")
        if ref is None:
            ref = x[0], st["itr"]
            continue
        err = float(np.abs(x - ref[0]).max() / np.abs(ref[0]).max())
        print(sD, copies, st["itr"], err, flush=True)
        assert st["itr"] == ref[1]
        assert err <= TOL
