"""The level launches, which serve rows of more than seven lower or upper blocks (no sweep task holds them), in every
storage precision, with wide and narrow column slices, one and several right-hand sides; and the sweep against the
dataflow kernels, which share nothing with it, on a full-size system.  Tolerances: the oracle's apply as in the
other apply tests (BF16 twice its distance from FP64, 3.5e-3); sweep and dataflow differ in the order of FP32 (or
FP64) sums of the same stored factor."""
import ctypes as C

import numpy as np
import pytest

import pyoracle as po
from chidg_amd.linsolve import Context, chidg_matrix, precon_ILU0
from chidg_amd.pattern import from_rows, hex_box

pytestmark = pytest.mark.gpu
TOL = {"fp64": 1e-12, "fp32": 1e-5, "bf16": 7e-3}


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16"])
@pytest.mark.parametrize("n,slice_w", [(6, None), (40, None), (40, 8), (135, None), (135, 16)])
def test_rows_of_eight_blocks(ctx, monkeypatch, n, slice_w, precision):
    if slice_w:
        monkeypatch.setenv("CDG_APPLY_SLICE_W", str(slice_w))
    nrows = 11
    p = from_rows(n, [[(j, 0) for j in range(nrows) if j != i and max(i, j) >= 8] + [(i, 0)] for i in range(nrows)])
    r = np.random.default_rng(n)
    blocks = r.standard_normal((p.nnzb, n, n)) * (0.2 / np.sqrt(n))
    blocks[p.col == np.repeat(np.arange(nrows), np.diff(p.row_ptr))] += 2 * np.eye(n)
    A = chidg_matrix(p, ctx)
    A.store(blocks.reshape(-1))
    L, D = po.ilu0_factor(p, blocks.reshape(-1))
    V = r.standard_normal((3, p.vec_len))
    M = precon_ILU0(precision).init(A)
    M.update(A)
    Z = np.empty_like(V)
    for _ in range(14):                       # (no other form after many applies)
        z = M.apply(A, V[0])
    ctx._check(ctx.lib.cdg_prec_apply_multi(ctx.h, M.h, A.h, 3, V.ctypes.data_as(C.c_void_p),
                                            Z.ctypes.data_as(C.c_void_p)), "cdg_prec_apply_multi")
    for k in range(3):
        ref = np.asarray(po.ilu0_apply(p, blocks.reshape(-1), L, D, V[k])).ravel()
        assert np.linalg.norm(Z[k] - ref) <= TOL[precision] * np.linalg.norm(ref)
        assert np.array_equal(Z[k], M.apply(A, V[k]))
    assert np.array_equal(z, Z[0])
    M.tear_down()
    A.release()


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32", 1e-6), ("bf16", 1e-6)])
@pytest.mark.parametrize("dims,n", [((16, 16, 16), 135), ((31, 17, 13), 40), ((6, 5, 5), 320)])
def test_sweep_against_dataflow(ctx, dims, n, precision, tol):
    import torch
    A = chidg_matrix(hex_box(*dims, n), ctx)
    A.fill_synthetic(11, 1 / np.sqrt(n), 0.1 / np.sqrt(n))
    v = A.synthetic_vector(1, like=torch.empty(0, dtype=torch.float64, device="cuda:0"))
    z = []
    for schedule in ("levels", "dataflow"):
        M = precon_ILU0(precision, schedule=schedule).init(A)
        M.update(A)
        z.append(M.apply(A, v))
        M.tear_down()
    assert float(torch.linalg.norm(z[0] - z[1]) / torch.linalg.norm(z[1])) < tol
    A.release()
