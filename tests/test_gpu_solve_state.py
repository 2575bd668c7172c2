"""What a memLS solve leaves behind and takes over: the statistics of a solver
object after solves of another one on the same matrix handle.

The systems are test_gpu_schur's (4x4 blocks on small graphs, D = -G^T
blockwise, K near twice the identity).
"""
import numpy as np
import pytest

from test_gpu_schur import _system

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cfa():
    import crimsonflowsolver_amd as cfa
    if cfa.device_count() < 1:
        pytest.fail("no GPU visible: the HIP path must run here")
    return cfa


def _handle(cfa, rowptr, colptr, faces=0):
    n = rowptr.size - 1
    return cfa.memLS_LHS_CREATE(n, n, colptr.size, None, rowptr, colptr, faces)


def _ns(cfa, absTolGM, maxItr=1, relTolGM=0.1):
    return cfa.memLS_LS_CREATE(cfa.LS_TYPE_NS, relTol=1e-12, dimKry=20, maxItr=maxItr, relTolIn=[relTolGM, 0.1],
                               absTolIn=[absTolGM, 1e-10], maxItrIn=[1, 50])


def test_gmres_statistics_are_the_solvers_own(cfa):
    """A solve whose GMRES calls all end at once (residual below absTol) leaves
    the solver's GM norms as they were: zero in a new one, its last solve's in a
    used one.  With the momentum solution zero, the second outer iteration's
    Gram matrix has a zero column: singular, the statistics up to there set."""
    rowptr, colptr, val, A = _system(60, [(i, (i + k) % 60) for i in range(60) for k in (1, 2, 3)], 5)
    lhs = _handle(cfa, rowptr, colptr)
    R = np.asfortranarray(np.random.default_rng(1).standard_normal((4, 60)))
    used = _ns(cfa, 1e-10)
    cfa.memLS_SOLVE(lhs, used, 4, R.copy(order="F"), val)
    before = used.stats("GM")
    assert before["iNorm"] > 0 and before["itr"] > 0
    fresh = _ns(cfa, 1e30)
    cfa.memLS_SOLVE(lhs, fresh, 4, R.copy(order="F"), val)
    got = fresh.stats("GM")
    assert (got["iNorm"], got["fNorm"], got["itr"], got["suc"], got["dB"]) == (0, 0, 0, 0, 0)
    assert fresh.stats("RI")["iNorm"] == used.stats("RI")["iNorm"]
    two = _ns(cfa, 1e30, maxItr=2)
    with pytest.raises(cfa.CrimsonError) as e:
        cfa.memLS_SOLVE(lhs, two, 4, R.copy(order="F"), val)
    assert e.value.code == 7
    assert two.stats("RI")["iNorm"] == used.stats("RI")["iNorm"] and two.stats("CG")["itr"] > 0


def test_gmres_db_of_a_last_call_that_ends_at_once(cfa):
    """The second momentum solve of an outer iteration starts from Rm - G P, smaller
    than Rm; an absTol between the two ends it at once, and GM's dB is then 0."""
    n = 60
    rowptr, colptr, val, A = _system(n, [(i, (i + k) % n) for i in range(n) for k in (1, 2, 3)], 5)
    lhs = _handle(cfa, rowptr, colptr)
    d = np.abs(np.diag(A)).reshape(n, 4).T
    # a momentum residual in the range of G, which the pressure removes for the most part
    p = np.random.default_rng(2).standard_normal(n)
    G = A.reshape(n, 4, n, 4)[:, :3, :, 3]
    R = np.zeros((4, n), order="F")
    R[:3] = np.einsum("aib,b->ia", G, p)
    L = A.reshape(n, 4, n, 4)[:, 3, :, 3]
    R[3] = 0.6 * (L @ p)
    n1 = np.linalg.norm((R / np.sqrt(d))[:3])
    ls = _ns(cfa, 1e-10, relTolGM=0.9)
    cfa.memLS_SOLVE(lhs, ls, 4, R.copy(order="F"), val)
    n2 = ls.stats("GM")["iNorm"]
    print("norms", n1, n2)
    assert n2 < 0.85 * n1 and ls.stats("GM")["dB"] != 0
    # below 0.9 n1 the first call's target is relTol's either way, so that P is the same
    ls = _ns(cfa, 0.5 * (0.9 * n1 + n2), relTolGM=0.9)
    cfa.memLS_SOLVE(lhs, ls, 4, R.copy(order="F"), val)
    got = ls.stats("GM")
    assert abs(got["iNorm"] - n1) <= 1e-12 * n1
    assert got["suc"] == 0 and got["dB"] == 0


def _coupled(cfa, n=60, seed=5):
    """A ring of 60 nodes with two coupled faces of 10 and 15 nodes."""
    rowptr, colptr, val, _ = _system(n, [(i, (i + k) % n) for i in range(n) for k in (1, 2, 3)], seed)
    lhs = _handle(cfa, rowptr, colptr, 2)
    rng = np.random.default_rng(6)
    v = [rng.uniform(0.2, 1.0, (3, k)) for k in (10, 15)]
    for f, start in enumerate((4, 30)):
        cfa.memLS_BC_CREATE(lhs, f + 1, v[f].shape[1], 3, cfa.BC_TYPE_Neu, np.arange(start, start + v[f].shape[1]) + 1,
                            np.asfortranarray(v[f]))
    lhs.set_val(4, val)
    return lhs, v


def _solver(cfa):
    return cfa.memLS_LS_CREATE(cfa.LS_TYPE_NS, relTol=1e-5, dimKry=40, maxItr=6, relTolIn=[0.1, 0.1], maxItrIn=[2, 200])


def test_graph_after_solves_with_other_faces(cfa):
    """A captured solve with two coupled faces, replayed after plain solves with one of
    them and with both: accepted, and the plain solve's bits.  Replayed after a
    face moved to other nodes (as many of them): the plain solve's bits there."""
    import torch
    lhs, v = _coupled(cfa)
    rhs = torch.from_numpy(1e3 * np.random.default_rng(8).standard_normal((60, 4))).cuda()
    both, one = np.array([7.0, 4.0]), np.array([7.0, 0.0])

    def plain(res):
        x = rhs.clone()
        cfa.memLS_SOLVE_dev(lhs, _solver(cfa), 4, x, res=res)
        return x

    buf = torch.empty_like(rhs)
    graph = cfa.memLS_SOLVE_graph(lhs, _solver(cfa), 4, buf, res=both)

    def replay():
        buf.copy_(rhs)
        torch.cuda.synchronize()
        graph.launch()
        return buf.clone()

    want = plain(both)
    assert torch.equal(replay(), want)
    assert not torch.equal(plain(one), want)
    with pytest.raises(cfa.CrimsonError) as e:  # another set is coupled
        replay()
    assert e.value.code == 8
    assert torch.equal(plain(both), want)
    for _ in range(2):
        assert torch.equal(replay(), want)
    cfa.memLS_BC_CREATE(lhs, 2, 15, 3, cfa.BC_TYPE_Neu, np.arange(35, 50) + 1, np.asfortranarray(v[1]))
    moved = replay()
    assert torch.equal(moved, plain(both)) and not torch.equal(moved, want)
    assert torch.equal(replay(), moved)


def test_graph_after_solves_in_the_other_precision(cfa):
    """A captured FP64 solve, replayed after plain FP32 solves of the same handle."""
    import torch
    from crimsonflowsolver_amd import mesh as M
    from crimsonflowsolver_amd.timestep import ResistanceCylinder
    c = ResistanceCylinder(M.cylinder_mesh(5, 5, 8), params=cfa.form_params(), ls=_solver(cfa))
    y, ac = c.state()
    c.residual(y, ac, y, ac)
    rhs = c.res4.clone()
    c.lhs.set_precision(32)  # both precisions' planes are there from here on
    c.lhs.set_precision(64)

    def plain():
        x = rhs.clone()
        cfa.memLS_SOLVE_dev(c.lhs, _solver(cfa), 4, x, res=c.faceres)
        return x

    buf = rhs.clone()
    graph = cfa.memLS_SOLVE_graph(c.lhs, _solver(cfa), 4, buf, res=c.faceres)
    want = plain()
    for _ in range(2):
        c.lhs.set_precision(32)
        plain()
        c.lhs.set_precision(64)
        buf.copy_(rhs)
        torch.cuda.synchronize()
        graph.launch()
        assert torch.equal(buf, want)


def test_solves_of_one_handle_from_threads(cfa):
    """Three threads at once on one handle that has not solved before: with its
    Dirichlet face, without it, and replays of a captured solve with it.  Each
    result has the bits of the same call alone on a handle of its own."""
    import threading

    import torch
    n = 3000
    i = np.arange(n)
    rp = np.concatenate([[0], np.cumsum(np.full(n, 5))]).astype(np.int32) + 1
    cols = np.sort((i[:, None] + np.arange(-2, 3)) % n, axis=1)
    rng = np.random.default_rng(3)
    val = np.zeros((16, 5 * n), order="F")
    diag = (cols == i[:, None]).ravel()
    val[[0, 5, 10, 15]] = np.where(diag, 2.0, -0.1)
    key = {(a, b): a * 5 + k for a in range(n) for k, b in enumerate(cols[a])}
    tr = np.array([key[(b, a)] for a in range(n) for b in cols[a]])
    g = 0.2 * rng.uniform(-1, 1, (3, 5 * n))
    val[[3, 7, 11]] = g
    val[12:15] = -g[:, tr]
    rhs = torch.from_numpy(1e3 * rng.standard_normal((n, 4))).cuda()
    fixed = np.arange(0, n, 7)
    neu = np.arange(1, 400, 7)
    v = rng.uniform(0.2, 1.0, (3, neu.size))
    res = np.array([0.0, 3.0])

    def handle():
        lhs = _handle(cfa, rp, (cols.ravel() + 1).astype(np.int32), 2)
        cfa.memLS_BC_CREATE(lhs, 1, fixed.size, 3, cfa.BC_TYPE_Dir, fixed + 1, np.zeros((3, fixed.size), order="F"))
        cfa.memLS_BC_CREATE(lhs, 2, neu.size, 3, cfa.BC_TYPE_Neu, neu + 1, np.asfortranarray(v))
        lhs.set_val(4, val)
        return lhs

    def solve(lhs, incL):
        x = rhs.clone()
        torch.cuda.synchronize()
        cfa.memLS_SOLVE_dev(lhs, _solver(cfa), 4, x, incL=np.array(incL, np.int32), res=res)
        return x

    want = [solve(handle(), inc) for inc in ((1, 1), (0, 1), (1, 1))]
    assert not torch.equal(want[0], want[1])
    lhs = handle()
    buf = rhs.clone()
    graph = cfa.memLS_SOLVE_graph(lhs, _solver(cfa), 4, buf, incL=np.array([1, 1], np.int32), res=res)

    def replay():
        buf.copy_(rhs)
        torch.cuda.synchronize()
        graph.launch()
        return buf.clone()

    calls = [lambda: solve(lhs, (1, 1)), lambda: solve(lhs, (0, 1)), replay]
    got, failed = [[], [], []], []
    start = threading.Barrier(3)

    def work(k):
        try:
            start.wait()
            for _ in range(8):
                got[k].append(calls[k]())
        except Exception as e:  # reported below
            failed.append((k, e))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    for k in range(3):
        assert len(got[k]) == 8 and all(torch.equal(x, want[k]) for x in got[k]), k


def test_release_workspaces(cfa):
    """release_workspaces gives the kept memory back; solves and a captured
    solve give the same bits before and after."""
    import torch
    from crimsonflowsolver_amd import mesh as M
    from crimsonflowsolver_amd.timestep import ResistanceCylinder
    c = ResistanceCylinder(M.cylinder_mesh(20, 20, 60), params=cfa.form_params(), ls=_solver(cfa))
    y, ac = c.state()
    c.residual(y, ac, y, ac)
    rhs = c.res4.clone()

    def plain():
        x = rhs.clone()
        cfa.memLS_SOLVE_dev(c.lhs, _solver(cfa), 4, x, res=c.faceres)
        return x

    want = plain()
    buf = rhs.clone()
    graph = cfa.memLS_SOLVE_graph(c.lhs, _solver(cfa), 4, buf, res=c.faceres)
    free = torch.cuda.mem_get_info()[0]
    cfa.release_workspaces()
    # at least the basis, 3 N doubles a vector, 40 vectors
    assert torch.cuda.mem_get_info()[0] - free >= 40 * 3 * c.N * 8
    torch.cuda.synchronize()
    graph.launch()
    assert torch.equal(buf, want)
    for _ in range(2):
        assert torch.equal(plain(), want)
        cfa.release_workspaces()
        cfa.release_workspaces()


_FAIL_MALLOC = r"""
#include <dlfcn.h>
#include <stddef.h>
/* hipMalloc that fails for one size: the next `fail_times` calls with it */
size_t fail_size = 0;
int fail_times = 0, failed = 0;
int hipMalloc(void **p, size_t n) {
  static int (*real)(void **, size_t);
  if (!real) real = (int (*)(void **, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_NOLOAD | RTLD_LAZY), "hipMalloc");
  if (n == fail_size && fail_times > 0) {
    --fail_times;
    ++failed;
    return 2; /* hipErrorOutOfMemory */
  }
  return real(p, n);
}
"""

_FAIL_CHILD = r"""
import ctypes, sys
sys.modules["torch"] = None  # the library's own HIP runtime, behind the stand-in
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import crimsonflowsolver_amd as cfa
size, times, failed = (t.in_dll(fake, k) for t, k in ((ctypes.c_size_t, "fail_size"), (ctypes.c_int, "fail_times"),
                                                      (ctypes.c_int, "failed")))
n = 3000
i = np.arange(n)
cols = np.sort((i[:, None] + np.arange(-2, 3)) % n, axis=1)
rng = np.random.default_rng(3)
val = np.zeros((16, 5 * n), order="F")
val[[0, 5, 10, 15]] = np.where((cols == i[:, None]).ravel(), 2.0, -0.1)
key = {(a, b): a * 5 + k for a in range(n) for k, b in enumerate(cols[a])}
g = 0.2 * rng.uniform(-1, 1, (3, 5 * n))
val[[3, 7, 11]] = g
val[12:15] = -g[:, [key[(b, a)] for a in range(n) for b in cols[a]]]
R = np.asfortranarray(1e3 * rng.standard_normal((4, n)))
rp = (5 * np.arange(n + 1) + 1).astype(np.int32)


def handle():
    return cfa.memLS_LHS_CREATE(n, n, 5 * n, None, rp, (cols.ravel() + 1).astype(np.int32), 0)


def solve(lhs):
    ls = cfa.memLS_LS_CREATE(cfa.LS_TYPE_NS, relTol=1e-6, dimKry=30, maxItr=5, relTolIn=[0.01, 0.01], maxItrIn=[2, 200])
    x = R.copy(order="F")
    cfa.memLS_SOLVE(lhs, ls, 4, x, val)
    return x


def armed(lhs, nbytes, count):
    before = failed.value
    size.value, times.value = nbytes, count
    x = solve(lhs)
    times.value = 0
    assert failed.value == before + count, (failed.value, before, count)
    return x


columns, values = 9 * n * 2, 9 * n * 8  # the two-ring has 9 entries a row, within 2-byte offsets
A = handle()
want = solve(A)
cfa.release_workspaces()
scale = np.abs(want).max()
# the pattern's buffer, with nothing to give back, and the values', tried again after
# the new pattern's share of the handle has been given back
for nbytes, count in ((columns, 1), (values, 2)):
    B = handle()
    two = armed(B, nbytes, count)
    assert not np.array_equal(two, want) and np.abs(two - want).max() <= 1e-3 * scale, nbytes
    assert np.array_equal(solve(B), want), ("formed again", nbytes)
    cfa.release_workspaces()
solve(A)  # idle now
C = handle()
assert np.array_equal(armed(C, values, 1), want)  # A's workspace given back, the allocation made
assert np.array_equal(solve(A), want)
print("CHILD_OK", flush=True)
"""


def test_failed_allocations_of_the_complement(cfa, tmp_path):
    """hipMalloc failing for the Schur complement's buffers, in a process of its own with
    a stand-in in front of the runtime's: that solve takes the two passes, the next
    one forms the complement; with another handle's workspace idle, that is given
    back and the allocation made again.  Tolerance: both operators' solutions have
    residuals under 1e-6 of the right-hand side's (condition numbers under 1e2)."""
    import os
    import subprocess
    import sys
    src, lib, child = tmp_path / "fail.c", tmp_path / "fail.so", tmp_path / "child.py"
    src.write_text(_FAIL_MALLOC)
    child.write_text(_FAIL_CHILD)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(lib), str(src), "-ldl"], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, PYTHONPATH=root)
    out = subprocess.run([sys.executable, "-u", str(child), str(lib)], env=env, capture_output=True, text=True,
                         timeout=100)
    assert out.returncode == 0 and "CHILD_OK" in out.stdout, out.stdout[-2000:] + out.stderr[-2000:]
