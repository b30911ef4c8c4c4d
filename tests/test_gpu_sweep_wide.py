"""The sweep where its levels have more tasks than the GPU has compute units: two levels of a few hundred rows (every
row of the second half coupled to two or more of the first), the task shape and the units of several tasks that such
patterns take, with levels that are no multiple of a unit, one and several right-hand sides.  Against the oracle's
apply; tolerances of the other apply tests, BF16 twice its distance from FP64 (3.5e-3)."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as po
from chidg_amd.linsolve import Context, chidg_matrix, precon_ILU0
from chidg_amd.pattern import from_rows

pytestmark = pytest.mark.gpu
TOL = {"fp64": 1e-12, "fp32": 1e-5, "bf16": 7e-3}


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16"])
@pytest.mark.parametrize("n,half,links", [(1, 301, 2), (5, 262, 2), (16, 259, 2), (40, 261, 2), (41, 258, 2),
                                          (64, 257, 2), (135, 131, 2), (22, 300, 7), (32, 260, 7), (42, 260, 6)])
def test_two_wide_levels(ctx, n, half, links, precision):
    """(22, 32 and 42 with many links: the most local memory that a unit takes, 76 KB)"""
    rows = [[(half + (i + d) % half, 0) for d in range(links)] + [(i, 0)] for i in range(half)]
    rows += [sorted(((i - d) % half, 0) for d in range(links)) + [(half + i, 0)] for i in range(half)]
    p = from_rows(n, rows)
    r = np.random.default_rng(n)
    blocks = r.standard_normal((p.nnzb, n, n)) * (0.2 / np.sqrt(n))
    blocks[p.col == np.repeat(np.arange(p.nrows), np.diff(p.row_ptr))] += 2 * np.eye(n)
    A = chidg_matrix(p, ctx)
    A.store(blocks.reshape(-1))
    L, D = po.ilu0_factor(p, blocks.reshape(-1))
    V = r.standard_normal((8, p.vec_len))
    ref = [np.asarray(po.ilu0_apply(p, blocks.reshape(-1), L, D, v)).ravel() for v in V]
    M = precon_ILU0(precision).init(A)
    M.update(A)
    assert np.linalg.norm(M.apply(A, V[0]) - ref[0]) <= TOL[precision] * np.linalg.norm(ref[0])
    for k in (2, 5, 8):
        Z = np.empty((k, p.vec_len))
        ctx._check(ctx.lib.cdg_prec_apply_multi(ctx.h, M.h, A.h, k, V.ctypes.data_as(C.c_void_p),
                                                Z.ctypes.data_as(C.c_void_p)), "cdg_prec_apply_multi")
        for q in range(k):
            assert np.linalg.norm(Z[q] - ref[q]) <= TOL[precision] * np.linalg.norm(ref[q])
            assert np.array_equal(Z[q], M.apply(A, V[q]))
    M.tear_down()
    A.release()
