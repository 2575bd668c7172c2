"""The residual's VJP on balls of tets around one hub, whose row is at the edges of
the adjoint's node passes (16 and 20 neighbours staged per row, 24 records in
flight, places of 64 bits above 1,024 blocks), with and without the
acceleration's cotangent.

Tolerance: that of test_gpu_adjoint.py for the same comparison, central
differences of the oracle's residual: 1e-6 (steps of 1e-6 relative in y, 1e-5 in
the acceleration and mu, whose terms are small in the residual's rounding).  The two
variants sum the same terms and agree to 1e-13 normwise."""
import numpy as np
import pytest

from test_gpu_formation_rows import _ball, _csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [14, 15, 16, 19, 20, 1024])
def test_vjp_long_row(oracle_lib, n):
    import torch
    import crimsonflowsolver_amd as cfa
    ien, x = _ball(n)
    N = n + 1
    rng = np.random.default_rng(n)
    y = np.asfortranarray(rng.normal(size=(N, 4)) * np.array([10.0, 1.0, 1.0, 1.0]))
    ac = np.asfortranarray(rng.uniform(-20, 20, size=(N, 4)))
    w = np.asfortranarray(rng.normal(size=(N, 4)))
    colm, rowp = _csr(ien, N)
    form = cfa.ElmGMRInterior(ien, colm, rowp, N)
    F = lambda a: torch.from_numpy(np.ascontiguousarray(a.T)).cuda()
    ybar, ybar2, acbar = (torch.full((4, N), 9.0, dtype=torch.float64, device="cuda") for _ in range(3))
    mub = form.vjp(F(y), F(ac), F(x), F(w), ybar)
    mub2 = form.vjp_ac(F(y), F(ac), F(x), F(w), ybar2, acbar)
    ybar, ybar2, acbar = (t.cpu().numpy().T for t in (ybar, ybar2, acbar))
    assert np.abs(ybar - ybar2).max() <= 1e-13 * np.abs(ybar).max()
    assert abs(mub - mub2) <= 1e-13 * abs(mub)
    assert np.all(acbar[:, 3] == 0.0)

    def J(yy, aa, mu=0.04):
        r, _, _ = oracle_lib.elmgmr_interior(ien, yy, aa, x, colm, rowp, oracle_lib.make_params(mu=mu, lhs=0))
        return float(np.sum(w * r))

    for k in range(2):
        d = np.asfortranarray(rng.normal(size=y.shape))
        h = 1e-6 * np.abs(y).max() / np.abs(d).max()
        fd, an = (J(y + h * d, ac) - J(y - h * d, ac)) / (2 * h), float(np.sum(ybar * d))
        print(n, "y", fd, an)
        assert abs(fd - an) <= 1e-6 * abs(fd)
        d[:, 3] = 0.0
        h = 1e-5 * np.abs(ac).max() / np.abs(d).max()
        fd, an = (J(y, ac + h * d) - J(y, ac - h * d)) / (2 * h), float(np.sum(acbar * d))
        print(n, "ac", fd, an)
        assert abs(fd - an) <= 1e-6 * abs(fd)
    h = 1e-5 * 0.04
    fd = (J(y, ac, 0.04 + h) - J(y, ac, 0.04 - h)) / (2 * h)
    print(n, "mu", fd, mub)
    assert abs(fd - mub) <= 1e-6 * abs(fd)
