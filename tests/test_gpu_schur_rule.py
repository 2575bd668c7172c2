"""Where the NS solver forms its Schur complement on large graphs: one cylinder in
its own numbering and numbered at random, just past the sizes at which the
random numbering keeps the two passes (FP64 327,680 rows, FP32 65,536).  Which
operator a solve took shows in the device memory that its first solve keeps:
the complement's 65 entries a row are more than half of the difference.  The two
solutions, of different operators on the same system, agree to the solver's
tolerance (1e-6 of the residual; scaled condition numbers of some hundred: 1e-3).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,grid", [(64, (44, 44, 240)), (32, (26, 26, 120))])
def test_scattered_numbering_takes_two_passes(bits, grid):
    import torch
    import crimsonflowsolver_amd as cfa
    from crimsonflowsolver_amd import mesh as M
    m = M.cylinder_mesh(*grid)
    n = m.numnp
    assert n > (327680 if bits == 64 else 65536)
    y, ac = M.poiseuille_state(m, seed=5)
    ibc, _ = M.dirichlet_codes(m)
    fixed, out = np.nonzero(ibc)[0], np.nonzero(m.outlet & (ibc == 0))[0]
    nabi = m.nabi()[out]
    T = lambda a: torch.from_numpy(np.ascontiguousarray(np.asarray(a).T)).cuda()
    held, x = [], []
    for scattered in (False, True):
        new = np.random.default_rng(11).permutation(n) if scattered else np.arange(n)  # new number of each node
        old = np.argsort(new)
        ien = np.asfortranarray(new[m.ien - 1].astype(np.int32) + 1)
        colm, rowp = cfa.genadj(ien, n)
        form = cfa.ElmGMRInterior(ien, colm, rowp, n, iBC=ibc[old], params=cfa.form_params(precision=bits))
        lhs = cfa.memLS_LHS_CREATE(n, n, rowp.size, None, colm, rowp, 2)
        cfa.memLS_BC_CREATE(lhs, 1, fixed.size, 3, cfa.BC_TYPE_Dir, new[fixed] + 1, np.zeros((3, fixed.size), order="F"))
        cfa.memLS_BC_CREATE(lhs, 2, out.size, 3, cfa.BC_TYPE_Neu, new[out] + 1, np.asfortranarray(nabi.T))
        rhs = torch.zeros((n, 4), dtype=torch.float64, device="cuda")
        form.to_lhs(T(np.asfortranarray(y[old])), T(np.asfortranarray(ac[old])), T(np.asfortranarray(m.x[old])), rhs, lhs)
        form.bc3res(rhs, res4_layout=True)
        form.sync()
        ls = cfa.memLS_LS_CREATE(cfa.LS_TYPE_NS, relTol=1e-6 if bits == 64 else 1e-4, dimKry=40, maxItr=10,
                                 relTolIn=[0.01, 0.05], maxItrIn=[2, 2000])
        cfa.release_workspaces()
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        cfa.memLS_SOLVE_dev(lhs, ls, 4, rhs, res=np.array([0.0, 0.5]))
        held.append(free - torch.cuda.mem_get_info()[0])
        assert ls.RI["suc"] == 1
        x.append(rhs.cpu().numpy()[new])
        del form, lhs
    values = 65 * n * bits // 8
    print("held", held, "values", values)
    assert held[0] - held[1] > 0.5 * values
    assert np.linalg.norm(x[1] - x[0]) <= (1e-3 if bits == 64 else 1e-1) * np.linalg.norm(x[0])
