"""A matrix of no rows, which the library accepts: every call on it returns at once, a solve with x empty, no
iterations and residual 0, whatever ran before on the context (a large solve, so that the GPU's local memory is
not zero)."""
import numpy as np
import pytest

import pyoracle as po
from chidg_amd import _lib
from chidg_amd.linsolve import Context, chidg_matrix, chidg_mv, fgmres, precon_identity, precon_ILU0
from chidg_amd.pattern import Pattern
from helpers import synthetic_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("orth", ["CGS", "MGS"])
@pytest.mark.parametrize("precon", ["identity", "fp64", "bf16"])
def test_no_rows(precon, orth):
    ctx = Context(0)
    make = precon_identity if precon == "identity" else lambda: precon_ILU0(precon)
    p, blocks = synthetic_system(4, 4, 4, 1, seed=3)
    A = chidg_matrix(p, ctx)
    A.store(blocks)
    b = po.fill_vector(p.vec_len, 1)
    ls = fgmres(nkrylov=30, tol=0.0, rtol=1e-8, nmax=40, inner_fgmres=False, orthogonalization=orth)
    ls.solve(A, np.zeros_like(b), b, make())
    e = np.zeros(0, np.int32)
    E = chidg_matrix(Pattern(0, 8, np.zeros(1, np.int32), e, e, None), ctx)
    E.store(np.zeros(0))
    M = make().init(E)
    M.update(E)
    assert chidg_mv(E, np.zeros(1)).size == 0
    M.apply(E, np.zeros(1), out=np.zeros(1))
    for inner in (False, True):
        ls = fgmres(nkrylov=30, tol=0.0, rtol=1e-8, nmax=-1, inner_fgmres=inner, orthogonalization=orth)
        ls.solve(E, np.zeros(1), np.zeros(1), M)
        assert ls.niter == 0 and ls.residual_norm == 0.0
        ls.solve_multi(E, np.zeros((3, 0)), np.zeros((3, 0)), M)
        assert ls.niter == [0, 0, 0] and ls.residual_norm == [0.0, 0.0, 0.0]
    with pytest.raises(_lib.CdgError):
        fgmres(nkrylov=0, inner_fgmres=False).solve(E, np.zeros(1), np.zeros(1), M)
    M.tear_down()
    E.release()
    A.release()
    ctx.close()
