"""More right-hand sides than a launch has grid rows (65535), on a system of two rows."""
import numpy as np
import pytest

from chidg_amd.linsolve import Context, chidg_matrix, fgmres, precon_ILU0
from chidg_amd.pattern import from_rows

pytestmark = pytest.mark.gpu


def test_70000_vectors():
    ctx = Context(0)
    A = chidg_matrix(from_rows(1, [[(0, 0), (1, 0)], [(0, 0), (1, 0)]]), ctx)
    A.store(np.array([2.0, 0.5, -0.25, 3.0]))
    k = 70000
    B = np.random.default_rng(0).standard_normal((k, 2))
    X = np.empty_like(B)
    ls = fgmres(nkrylov=3, tol=0.0, rtol=1e-10, inner_fgmres=False)
    ls.solve_multi(A, X, B, precon_ILU0())
    ref = np.linalg.solve(np.array([[2.0, 0.5], [-0.25, 3.0]]), B.T).T     # ILU(0) of two rows is their LU
    assert np.abs(X - ref).max() <= 1e-13 * np.abs(ref).max()
    assert set(ls.niter) == {1} and ls.stats[0].factored == 1
    A.release()
    ctx.close()
