"""The apply where no row has lower or upper blocks (block Jacobi, block-diagonal patterns, k_diag): sizes around its
256 threads and 16 columns in flight, one and several right-hand sides, a batch with uneven ones, in place.
z = Dinv v over the stored values in FP64 sums: within n roundings of FP64 (320 x 1.1e-16 < 1e-13)."""
import ctypes as C

import numpy as np
import pytest
import torch

from chidg_amd.linsolve import Context, batch, chidg_matrix, fgmres, precon_ILU0, precon_jacobi
from chidg_amd.pattern import from_rows, hex_box

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def system(ctx, p, seed):
    r = np.random.default_rng(seed)
    blocks = r.standard_normal((p.nnzb, p.n, p.n)) * (0.3 / np.sqrt(p.n))
    blocks[p.col == np.repeat(np.arange(p.nrows), np.diff(p.row_ptr))] += 2 * np.eye(p.n)
    A = chidg_matrix(p, ctx)
    A.store(blocks.reshape(-1))
    return A


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16"])
@pytest.mark.parametrize("kind,n,nrows", [("diag", *q) for q in [
    (1, 1), (1, 257), (3, 170), (5, 52), (8, 100), (15, 40), (16, 33), (17, 31), (64, 9), (127, 5), (128, 5), (129, 4),
    (135, 7), (255, 3), (257, 3), (320, 3)]] + [("jacobi", 5, 12), ("jacobi", 135, 12)])
def test_diag(ctx, kind, n, nrows, precision):
    p = from_rows(n, [[(i, 0)] for i in range(nrows)]) if kind == "diag" else hex_box(4, 3, 1, n, periodic=(True, True, False))
    A = system(ctx, p, n)
    M = (precon_ILU0 if kind == "diag" else precon_jacobi)(precision).init(A)
    M.update(A)
    D = np.asarray(M.factors(A)[1]).reshape(-1, n, n).transpose(0, 2, 1)
    V = np.random.default_rng(n).standard_normal((11, p.vec_len))
    ref = [np.einsum("irc,ic->ir", D, v.reshape(-1, n)).ravel() for v in V]
    for k in (1, 2, 3, 8, 11):
        Z = np.empty((k, p.vec_len))
        ctx._check(ctx.lib.cdg_prec_apply_multi(ctx.h, M.h, A.h, k, V.ctypes.data_as(C.c_void_p),
                                                Z.ctypes.data_as(C.c_void_p)), "cdg_prec_apply_multi")
        for r in range(k):
            assert rel(Z[r], ref[r]) < 1e-13
            assert np.array_equal(Z[r], M.apply(A, V[r]))
    w = torch.from_numpy(V[0]).to("cuda:0")
    torch.cuda.synchronize()
    M.apply_async(A, w, w, order=False)
    torch.cuda.synchronize()
    assert np.array_equal(w.cpu().numpy(), M.apply(A, V[0]))
    M.tear_down()
    A.release()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_solves(ctx, precision):
    """Block-diagonal systems: FGMRES ends after one step (two where Dinv is FP32) with the direct solution; in a
    batch with uneven right-hand sides as alone."""
    n, rows = 24, (5, 12)
    mats = [system(ctx, from_rows(n, [[(i, 0)] for i in range(m)]), m) for m in rows]
    bt = batch(mats, [3, 1], precision=precision, nkrylov=8)
    r = np.random.default_rng(5)
    B = [torch.from_numpy(r.standard_normal((k, m * n))).cuda() for k, m in zip((3, 1), rows)]
    X = [torch.empty_like(b) for b in B]
    bt.solve(B, X, rtol=1e-10)
    for A, b, x in zip(mats, B, X):
        d = A.to_host().reshape(-1, n, n).transpose(0, 2, 1)
        for q in range(len(b)):
            ref = np.linalg.solve(d, b[q].cpu().numpy().reshape(-1, n, 1)).ravel()
            assert rel(x[q].cpu().numpy(), ref) < 1e-9
            ls = fgmres(nkrylov=8, tol=0.0, rtol=1e-10, inner_fgmres=False)
            y = np.zeros(A.vec_len)
            ls.solve(A, y, b[q].cpu().numpy(), precon_ILU0(precision))
            assert rel(y, ref) < 1e-9 and 1 <= ls.niter <= 3
    bt.close()
