"""Batches on resident teams at the sizes where the layout changes: one and two
systems (larger teams), more systems than teams, sizes that need a larger team
or no team at all, 1 to 4 right-hand sides, systems that converge at once, in
2D and 3D.

Reference: the explicit layout (8 threads per row, 512 rows per tile), which
iterates by separate launches.  Both stop at 1e-12, so their solutions differ by
at most the two residuals times the condition of the problem: a few 1e-12 times
1e3 to 1e4 here; the bar is 1e-8 as for the other batch tests.  After a fixed
number of iterations (25) only rounding separates them: 25 * 400 eps = 1.1e-12,
the bar ten times that.
"""
import numpy as np
import pytest

from pigfem_assignment_amd import batch, configs, _lib as L
from pigfem_assignment_amd.api import DeviceContext, HostProblem

pytestmark = pytest.mark.gpu


def _rves(sizes):
    out = []
    for i, n in enumerate(sizes):
        incl = configs.rsa(2, 0.12, 0.16, 2, gap=min(2.0 / n, 0.1), seed=i + 1)
        out.append(batch.periodic_rve_problem(n, 0, inclusions=incl)[0])
    return out


def _cubes(sizes):
    bcs = [(L.SET_LEFT, 0, d, 0.0) for d in range(3)] + [(L.SET_RIGHT, 0, 0, 0.01)]
    return [HostProblem("tet4", (n,) * 3, (0,) * 3, (1,) * 3, inclusions=[[1, 0.5, 0.5, 0.5, 0.3]] if n > 4 else (),
                        materials=(configs.MATRIX, configs.INCLUSION), bcs=bcs) for n in sizes]


@pytest.mark.parametrize("parts", ["2d:40", "2d:32,33", "2d:20,64,24,48,36,52,28,44,30,34,22", "2d:300,24",
                                   "2d:24,24,24,24,24,24,24,24,24,24,24,24,24,24,24,24,24,24,160", "3d:9,14,5", "3d:30,8"])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 4])
def test_teams_match_launches(parts, nrhs):
    kind, sizes = parts.split(":")
    sizes = [int(n) for n in sizes.split(",")]
    B = batch.BatchProblem(_rves(sizes) if kind == "2d" else _cubes(sizes))
    ctx = DeviceContext(B)
    ctx.assemble(L.PGF_ASM_JAC)
    F = np.random.RandomState(nrhs).standard_normal((nrhs, B.n_free))
    F[-1, B.sys_ptr[0]: B.sys_ptr[1]] = 0.0  # one pair with nothing to solve
    for again in range(2):  # laid out, then laid out already
        X, its, rel, ms, tune = ctx.batch_pcg(B.sys_ptr, F, rtol=1e-30, maxit=25)
        R, rits, rrel, rms, _ = ctx.batch_pcg(B.sys_ptr, F, rtol=1e-30, maxit=25, tune=(8, 512))
        assert np.array_equal(its, rits) and its[0, -1] == 0 and its.max() == (25 if np.any(F) else 0)
        err = np.max(np.abs(X - R)) / max(np.max(np.abs(R)), 1e-300)  # (a lone zero pair stays zero)
        print("%s nrhs %d: 25 iterations, err %.1e" % (parts, nrhs, err), flush=True)
        assert err <= 1.1e-11 and np.allclose(rel, rrel, rtol=1e-9)
    X, its, rel, ms, tune = ctx.batch_pcg(B.sys_ptr, F, rtol=1e-12)
    R, rits, rrel, rms, _ = ctx.batch_pcg(B.sys_ptr, F, rtol=1e-12, tune=(8, 512))
    print("%s nrhs %d: teams %.2f ms, launches %.2f ms, choice %s" % (parts, nrhs, ms, rms, tune), flush=True)
    assert np.all(rel <= 1e-12) and np.max(np.abs(its - rits)) <= 0.05 * rits.max() + 5
    for s in range(len(sizes)):
        sl = slice(B.sys_ptr[s], B.sys_ptr[s + 1])
        assert np.max(np.abs(X[:, sl] - R[:, sl])) <= 1e-8 * np.max(np.abs(R[:, sl]))


def test_systems_that_couple_are_refused():
    B = batch.BatchProblem(_rves([24, 32]))
    ctx = DeviceContext(B)
    ctx.assemble(L.PGF_ASM_JAC)
    F = np.ones((1, B.n_free))
    wrong = B.sys_ptr.copy()
    wrong[1] -= 2
    for _ in range(2):
        with pytest.raises(RuntimeError, match="couples two systems"):
            ctx.batch_pcg(wrong, F)
        ctx.batch_pcg(B.sys_ptr, F, rtol=1e-6)
    # the same rows as one system
    X, its, rel, ms, _ = ctx.batch_pcg(B.sys_ptr[[0, 2]], F, rtol=1e-10)
    assert np.all(rel <= 1e-10)
