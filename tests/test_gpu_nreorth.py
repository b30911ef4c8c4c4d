"""The count of re-orthogonalized steps that a solve reports: the outer solver's and its nested solver's together.
Against the same nested FGMRES (type_fgmres.f90:81-310) in numpy; no step's test is closer to its threshold than
1e-6, so that rounding cannot change a count."""
import numpy as np
import pytest

from chidg_amd.linsolve import Context, chidg_matrix, fgmres, precon_identity
from chidg_amd.pattern import from_rows

pytestmark = pytest.mark.gpu


def plain(A, b, m, tol, rtol, nmax, orth, inner, seen):
    """x of the (nested) FGMRES with the identity as preconditioner; seen: the criterion of every step."""
    x = np.zeros_like(b)
    niter, res, r00 = 0, np.inf, None
    while res > tol:
        r = b - A @ x
        beta = np.linalg.norm(r)
        r00 = beta if r00 is None else r00
        V, Z, H = [r / beta], [], np.zeros((m + 1, m))
        for j in range(m):
            z = V[j].copy()
            if inner:
                z = z + plain(A, V[j] - A @ z, *inner, None, seen)
            Z.append(z)
            w = A @ z
            nb = np.linalg.norm(w)
            for second in range(2):
                if orth == "CGS":
                    h = np.array([v @ w for v in V])
                    w = w - np.array(V).T @ h
                    H[:j + 1, j] += h
                else:
                    for i, v in enumerate(V):
                        h = v @ w
                        w = w - h * v
                        H[i, j] += h
                if second == 0:
                    seen.append(np.abs(H[:j + 1, j]).sum() / nb)
                    if seen[-1] < 1:
                        break
            H[j + 1, j] = np.linalg.norm(w)
            V.append(w / H[j + 1, j])
            e = np.zeros(j + 2)
            e[0] = beta
            y = np.linalg.lstsq(H[:j + 2, :j + 1], e, rcond=None)[0]
            res = np.linalg.norm(H[:j + 2, :j + 1] @ y - e)
            niter += 1
            if res < tol or res / r00 < rtol or niter >= nmax > 0:
                return x + np.array(Z).T @ y
        x = x + np.array(Z).T @ y
    return x


@pytest.mark.parametrize("orth", ["CGS", "MGS"])
@pytest.mark.parametrize("inner", [False, True])
def test_counts(inner, orth):
    n, rows = 6, 7
    p = from_rows(n, [[(j, 0) for j in range(rows) if j != i] + [(i, 0)] for i in range(rows)])
    r = np.random.default_rng(4)
    blocks = r.standard_normal((p.nnzb, n, n)) * 0.2
    blocks[p.col == np.repeat(np.arange(rows), np.diff(p.row_ptr))] += 1.5 * np.eye(n)
    full = np.zeros((rows, n, rows, n))
    for i in range(rows):
        for b in range(p.row_ptr[i], p.row_ptr[i + 1]):
            full[i, :, p.col[b], :] = blocks[b].T
    b = r.standard_normal(rows * n)
    kw = dict(nkrylov=12, tol=0.0, rtol=1e-6, nmax=9)
    nested = (4, 0.0, 1e-3, 6, orth) if inner else None
    seen = []
    plain(full.reshape(rows * n, rows * n), b, *kw.values(), orth, nested, seen)
    assert min(abs(c - 1) for c in seen) > 1e-6 and any(c >= 1 for c in seen) and any(c < 1 for c in seen)
    ctx = Context(0)
    A = chidg_matrix(p, ctx)
    A.store(blocks.reshape(-1))
    ls = fgmres(**kw, orthogonalization=orth, inner_fgmres=inner)
    if inner:
        ls.inner_nkrylov, ls.inner_tol, ls.inner_rtol, ls.inner_nmax, ls.inner_orthogonalization = nested
    M = precon_identity()
    for _ in range(2):                        # counted per solve
        ls.solve(A, np.zeros_like(b), b, M)
        assert ls.stats.nreorth == sum(c >= 1 for c in seen)
    A.release()
    ctx.close()
