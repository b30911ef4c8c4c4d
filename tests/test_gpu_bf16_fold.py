"""BF16-stored ILU(0): the two operators of its apply, entry by entry.  The plain sweep's is L, U and Dinv, each
rounded to BF16; the folded sweep's is L, Dinv and W = Dinv U, rounded once from the FP32 Dinv (the row-slice and
stream schedules, several vectors, a batch, and the default schedule once a factor has served 12 applies).  Each is
applied here in FP64 with the stored values.  What is left between that and the GPU's apply is FP32 sums (1e-6) and
the entries of W that the FP32 Dinv's error (1e-6 of itself) rounds the other way: one in a thousand by one BF16
step, at most 5e-5 of the result in a simulation of these systems.  The two operators differ by 1e-3 to 4e-3
there; the bound is between."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as po
from chidg_amd.linsolve import Context, batch, chidg_matrix, precon_ILU0
from chidg_amd.pattern import from_rows, hex_box

TOL = 3e-4


def bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return ((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32).view(np.float32).astype(np.float64)


def system(p, seed):
    r = np.random.default_rng(seed)
    blocks = r.standard_normal((p.nnzb, p.n, p.n)) * (0.8 / np.sqrt(p.n))
    diag = p.col == np.repeat(np.arange(p.nrows), np.diff(p.row_ptr))
    blocks[diag & (p.kind == 0)] += 2 * np.eye(p.n)
    return blocks


def local(p, i):
    """(column, block) of row i's lower and upper entries."""
    e = [(int(p.col[b]), b) for b in range(p.row_ptr[i], p.row_ptr[i + 1]) if p.kind[b] == 0]
    return [q for q in e if q[0] < i], [q for q in e if q[0] > i]


def apply_ref(p, blocks, L, D, D_fold, v):
    """z = M^-1 v; L and D as stored, D_fold: None, or the Dinv of W.  Column-major blocks."""
    B = blocks.transpose(0, 2, 1)
    Lm, Dm = L.reshape(-1, p.n, p.n).transpose(0, 2, 1), D.reshape(-1, p.n, p.n).transpose(0, 2, 1)
    y = v.reshape(-1, p.n).copy()
    for i in range(p.nrows):
        for j, b in local(p, i)[0]:
            y[i] -= Lm[b] @ y[j]
    z = np.zeros_like(y)
    for i in reversed(range(p.nrows)):
        up = local(p, i)[1]
        if D_fold is None:
            z[i] = Dm[i] @ (y[i] - sum((bf16(B[b]) @ z[k] for k, b in up), np.zeros(p.n)))
        else:
            Di = D_fold.reshape(-1, p.n, p.n)[i].T
            z[i] = Dm[i] @ y[i] - sum((bf16(Di @ B[b]) @ z[k] for k, b in up), np.zeros(p.n))
    return z.ravel()


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def wide_rows(n, nrows, reach, seed):
    """Rows coupled to up to `reach` earlier rows, symmetric pattern, at most `reach` later ones."""
    r = np.random.default_rng(seed)
    lower, nup = [set() for _ in range(nrows)], np.zeros(nrows, int)
    for i in range(1, nrows):
        for j in r.permutation(i)[:int(r.integers(0, reach + 1))]:
            if nup[j] < reach:
                lower[i].add(int(j))
                nup[j] += 1
    return from_rows(n, [[(j, 0) for j in sorted(lower[i])] + [(j, 0) for j in range(i + 1, nrows) if i in lower[j]] +
                         [(i, 0)] for i in range(nrows)])


PATTERNS = [(1, 40, 3), (5, 30, 6), (8, 24, 4), (40, 20, 3), (40, 18, 6), (135, 8, 3), (136, 8, 5), (193, 6, 3),
            (320, 6, 3), (320, 7, 6)]


@pytest.mark.parametrize("n,nrows,reach", [q for q in PATTERNS if q[0] <= 40])
def test_bound_lies_between(n, nrows, reach):
    """On the CPU: the operators are further apart than the bound, the FP32 Dinv's error moves W by less."""
    p = wide_rows(n, nrows, reach, n + reach)
    blocks = system(p, 3)
    L, D = (np.asarray(a).ravel() for a in po.ilu0_factor(p, blocks.ravel()))
    r = np.random.default_rng(1)
    v = r.standard_normal(p.vec_len)
    fold = apply_ref(p, blocks, bf16(L), bf16(D), D, v)
    near = apply_ref(p, blocks, bf16(L), bf16(D), D * (1 + 1e-6 * r.standard_normal(D.shape)), v)
    assert rel(near, fold) < TOL / 5
    assert rel(apply_ref(p, blocks, bf16(L), bf16(D), None, v), fold) > 3 * TOL


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


def both(ctx, p, seed, v):
    """(A, the plain operator's apply, the folded one's) of a system on the device."""
    blocks = system(p, seed)
    A = chidg_matrix(p, ctx)
    A.store(blocks.reshape(-1))
    M = precon_ILU0("bf16").init(A)
    M.update(A)
    L, D = (np.asarray(a).ravel() for a in M.factors(A))
    M.tear_down()
    D64 = np.asarray(po.ilu0_factor(p, blocks.ravel())[1]).ravel()
    return A, [apply_ref(p, blocks, L, D, None, w) for w in v], [apply_ref(p, blocks, L, D, D64, w) for w in v]


def multi(ctx, M, A, V):
    Z = np.empty_like(V)
    ctx._check(ctx.lib.cdg_prec_apply_multi(ctx.h, M.h, A.h, len(V), V.ctypes.data_as(C.c_void_p),
                                            Z.ctypes.data_as(C.c_void_p)), "cdg_prec_apply_multi")
    return Z


@pytest.mark.gpu
@pytest.mark.parametrize("n,nrows,reach", PATTERNS)
def test_operators(ctx, n, nrows, reach):
    p = wide_rows(n, nrows, reach, n + reach)
    V = np.random.default_rng(n).standard_normal((11, p.vec_len))
    A, plain, fold = both(ctx, p, 3, V)
    for schedule, ref in (("levels", plain), ("auto", plain), ("rowslice", fold), ("stream", fold)):
        M = precon_ILU0("bf16", schedule=schedule).init(A)
        M.update(A)
        for k in range(2):
            assert rel(M.apply(A, V[k]), ref[k]) < TOL, schedule
        M.tear_down()
    M = precon_ILU0("bf16").init(A)
    M.update(A)
    for k in (2, 3, 8, 11):
        Z = multi(ctx, M, A, V[:k].copy())
        for r in range(k):
            assert rel(Z[r], fold[r]) < TOL, (k, r)
    M.tear_down()
    A.release()


@pytest.mark.gpu
def test_default_schedule(ctx):
    """From the 13th apply on, or from the first when the last factor served more; counted per factor, and a
    12-step solve counts 12.  Applies of a solve count like applies on their own."""
    from chidg_amd.linsolve import fgmres
    p = hex_box(4, 3, 3, 40)
    V = np.random.default_rng(0).standard_normal((1, p.vec_len))
    A, (plain,), (fold,) = both(ctx, p, 5, V)
    M = precon_ILU0("bf16").init(A)

    def served(first, count):
        M.update(A)
        got = [M.apply(A, V[0]) for _ in range(count)]
        assert all(rel(z, plain) < TOL for z in got[:first]) and all(rel(z, fold) < TOL for z in got[first:])

    served(12, 14)
    served(0, 5)
    served(12, 12)
    served(12, 13)
    M.update(A)
    M.update(A)
    ls = fgmres(nkrylov=30, tol=0.0, rtol=1e-30, nmax=12, inner_fgmres=False)
    x = np.zeros(p.vec_len)
    ls.solve(A, x, V[0], M)          # factors, 12 steps
    assert ls.niter == 12
    served(12, 12)
    ls = fgmres(nkrylov=5, tol=0.0, rtol=1e-30, nmax=13, inner_fgmres=False)
    ls.solve(A, x, V[0], M)
    assert ls.niter == 13
    served(0, 2)
    M.tear_down()
    A.release()


@pytest.mark.gpu
def test_capture_and_update(ctx):
    """A captured folded apply follows an update on replay, whether W was formed before the capture or in it; the
    allocation-free entry gives the same bits."""
    import torch
    p = wide_rows(40, 20, 3, 9)
    V = np.random.default_rng(1).standard_normal((1, p.vec_len))
    v = torch.from_numpy(V[0]).to("cuda:0")
    s = torch.cuda.ExternalStream(ctx.stream_ptr())
    for before in (True, False):
        A, _, (fold,) = both(ctx, p, 5, V)
        M = precon_ILU0("bf16", schedule="rowslice").init(A)
        M.update(A)
        z, w = torch.zeros_like(v), torch.zeros_like(v)
        if before:
            M.apply(A, v, out=z)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            M.apply_async(A, v, z, order=False)
        graph.replay()
        torch.cuda.synchronize()
        assert rel(z.cpu().numpy(), fold) < TOL
        A2, _, (fold2,) = both(ctx, p, 6, V)
        A2.release()
        A.store(system(p, 6).reshape(-1))
        M.update(A)
        for _ in range(3):
            z.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert rel(z.cpu().numpy(), fold2) < TOL
            assert torch.equal(M.apply(A, v), z)
        code = ctx.lib.cdg_prec_apply_noalloc(ctx.h, M.h, A.h, C.c_void_p(v.data_ptr()), C.c_void_p(w.data_ptr()))
        torch.cuda.synchronize()
        assert code == 0 and torch.equal(w, z)
        M.tear_down()
        A.release()


@pytest.mark.gpu
def test_batch_takes_w(ctx):
    """One step of a batch's solves: x = c M^-1 b, so its direction is the folded apply's; again after an update."""
    p = hex_box(3, 3, 2, 40)
    V = np.random.default_rng(2).standard_normal((3, p.vec_len))
    A, _, fold = both(ctx, p, 7, V)
    import torch
    bt = batch([A, A], [1, 3], precision="bf16", nkrylov=4)
    B = [torch.from_numpy(V[:1].copy()).cuda(), torch.from_numpy(V.copy()).cuda()]
    for seed in (7, 8):
        if seed == 8:
            A.store(system(p, 8).reshape(-1))
            bt.update([A, A])
            A2, _, fold = both(ctx, p, 8, V)
            A2.release()
        X = [torch.empty_like(b) for b in B]
        bt.solve(B, X, tol=0.0, rtol=1e-30, nmax=1)
        for s in (0, 1):
            for r in range(len(B[s])):
                x, f = X[s][r].cpu().numpy(), fold[r]
                assert rel(x * (f @ x) / (x @ x), f) < TOL
    bt.close()
    A.release()
