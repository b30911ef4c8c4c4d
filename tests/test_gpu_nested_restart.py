"""A nested FGMRES whose inner solver restarts (its Krylov space is smaller than the steps it needs), against the
oracle's nested solve; and a solve after it, which counts its own restarts only."""
import numpy as np
import pytest

import pyoracle as po
from chidg_amd.linsolve import Context, chidg_matrix, fgmres, precon_ILU0
from helpers import synthetic_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("orth", ["CGS", "MGS"])
@pytest.mark.parametrize("nkrylov,inner_nkrylov", [(30, 1), (30, 2), (3, 2)])
def test_inner_restarts(nkrylov, inner_nkrylov, orth):
    p, blocks = synthetic_system(4, 4, 2, 1, seed=29, s_off_scale=0.6)
    b = po.fill_vector(p.vec_len, 3)
    kw = dict(nkrylov=nkrylov, tol=0.0, rtol=1e-9, nmax=-1, orthogonalization=orth, inner_fgmres=True,
              inner_nkrylov=inner_nkrylov, inner_tol=1e-30, inner_rtol=1e-2, inner_nmax=9, inner_orthogonalization=orth)
    ref, niter, _, _ = po.fgmres(p, blocks, b, **kw)
    ctx = Context(0)
    A = chidg_matrix(p, ctx)
    A.store(blocks)
    ls, M = fgmres(**kw), precon_ILU0()
    for _ in range(2):
        x = np.zeros_like(b)
        ls.solve(A, x, b, M)
        assert abs(ls.niter - niter) <= 1
        assert ls.stats.nrestart == (ls.niter - 1) // nkrylov
        assert np.linalg.norm(x - ref) <= 1e-7 * np.linalg.norm(ref)
    M.tear_down()
    A.release()
    ctx.close()
