"""A sweep that gives up waiting (forced from the host: CDG_RS_SPIN=1, one poll a wait) is reported by the call, or
the next call, on its own preconditioner or batch, and by no other."""
import numpy as np
import pytest
import torch

import pyoracle as po
from chidg_amd import _lib
from chidg_amd.linsolve import Context, batch, chidg_matrix, fgmres, precon_ILU0
from helpers import synthetic_system

pytestmark = pytest.mark.gpu


@pytest.fixture
def parts(monkeypatch):
    ctx = Context(0)
    p, blocks = synthetic_system(4, 4, 4, 1, seed=17)
    A = chidg_matrix(p, ctx)
    A.store(blocks)
    good = precon_ILU0().init(A)
    good.update(A)
    v = po.fill_vector(p.vec_len, 3)
    ref = good.apply(A, v)

    def impatient(make):                      # plans made within it poll once
        monkeypatch.setenv("CDG_RS_SPIN", "1")
        made = make()
        monkeypatch.delenv("CDG_RS_SPIN")
        return made

    yield ctx, A, good, v, ref, impatient
    A.release()
    ctx.close()


def right(good, A, v, ref):
    assert np.array_equal(good.apply(A, v), ref)
    x = np.zeros_like(v)
    ls = fgmres(nkrylov=30, tol=0.0, rtol=1e-8, inner_fgmres=False)
    ls.solve(A, x, v, good)
    X = np.zeros((2, v.size))
    ls.solve_multi(A, X, np.stack([v, v]), good)
    assert np.array_equal(X[0], x)


def test_queued_apply(parts):
    ctx, A, good, v, ref, impatient = parts
    bad = impatient(lambda: precon_ILU0().init(A))
    bad.update(A)
    w = torch.from_numpy(v).to("cuda:0")
    z = torch.empty_like(w)
    for _ in range(20):                       # (one call may find every value ready)
        bad.apply_async(A, w, z, order=False)
    torch.cuda.synchronize()
    right(good, A, v, ref)
    with pytest.raises(_lib.CdgError, match="gave up"):
        bad.apply(A, v)
    bad.tear_down()
    right(good, A, v, ref)
    again = precon_ILU0()                     # takes the word that `bad` gave back
    again.init(A)
    again.update(A)
    again.tear_down()
    right(good, A, v, ref)


def test_solve(parts):
    ctx, A, good, v, ref, impatient = parts
    bad = impatient(lambda: precon_ILU0().init(A))
    x = np.zeros_like(v)
    with pytest.raises(_lib.CdgError, match="gave up"):
        for _ in range(5):
            fgmres(nkrylov=30, tol=0.0, rtol=1e-8, inner_fgmres=False).solve(A, x, v, bad)
    right(good, A, v, ref)
    bad.tear_down()


def test_batch(parts):
    ctx, A, good, v, ref, impatient = parts
    bt = impatient(lambda: batch([A, A], [1, 2], precision="fp32", nkrylov=30))
    B = [torch.from_numpy(v[None].copy()).cuda(), torch.from_numpy(np.stack([v, 2 * v])).cuda()]
    X = [torch.empty_like(b) for b in B]
    with pytest.raises(_lib.CdgError, match="gave up"):
        for _ in range(5):
            bt.solve(B, X)
    right(good, A, v, ref)
    bt.close()
    right(good, A, v, ref)
