"""Sums over a team at the team sizes where their layout changes: one block (no
exchange), two, the blocks one load reads (8 for six and eight values, 16 for
four, 32 for two) and one more, one pass of loads (128) and more, nearly all;
1 to 4 right-hand sides are sums of 1, 2, 3, 4, 6 and 8 values.

Reference: the explicit layout, which iterates by separate launches.  After 25
iterations only rounding separates them: 25 * 400 eps = 1.1e-12; the bar is ten
times that.  The iteration counts and residuals are the same.
"""
import numpy as np
import pytest

from pigfem_assignment_amd import batch, configs, _lib as L
from pigfem_assignment_amd.api import DeviceContext

pytestmark = pytest.mark.gpu


# an n x n periodic cell has about n^2 groups of rows, 128 of them a block
@pytest.mark.parametrize("n", [10, 16, 32, 33, 45, 46, 63, 65, 90, 91, 127, 128, 131, 180])
def test_sums_match_launches(n):
    incl = configs.rsa(2, 0.12, 0.16, 2, gap=min(2.0 / n, 0.1), seed=n)
    B = batch.BatchProblem([batch.periodic_rve_problem(n, 0, inclusions=incl)[0]])
    ctx = DeviceContext(B)
    ctx.assemble(L.PGF_ASM_JAC)
    for nrhs in (1, 2, 3, 4):
        F = np.random.RandomState(nrhs).standard_normal((nrhs, B.n_free))
        X, its, rel, _, _ = ctx.batch_pcg(B.sys_ptr, F, rtol=1e-30, maxit=25)
        R, rits, rrel, _, _ = ctx.batch_pcg(B.sys_ptr, F, rtol=1e-30, maxit=25, tune=(8, 512))
        err = np.max(np.abs(X - R)) / np.max(np.abs(R))
        print("%d x %d, %d right-hand sides: err %.1e" % (n, n, nrhs, err), flush=True)
        assert np.array_equal(its, rits) and np.allclose(rel, rrel, rtol=1e-9)
        assert err <= 1.1e-11
