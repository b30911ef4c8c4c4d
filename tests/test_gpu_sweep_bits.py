"""The sweep's sums under FP32 and BF16 storage: a task's base and the values it passes on are FP64, so a result that
is a small difference of FP64 inputs keeps its digits.  Two rows coupled by identities (all products exact):
y_0 = v_0, z_1 = v_1 - 1 = 1, z_0 = v_0 - z_1 with v_0 = 1 + d, |d| about 1e-9.  z_0 is narrowed to FP32 once, for the
product with Dinv_0 = I (6e-8 of itself); 1 + d itself is rounded at 1e-16, 2e-7 of d.  Values passed on in FP32
would leave nothing of d."""
import ctypes as C

import numpy as np
import pytest

from chidg_amd.linsolve import Context, chidg_matrix, precon_ILU0
from chidg_amd.pattern import from_rows

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("precision", ["fp32", "bf16"])
@pytest.mark.parametrize("n", [1, 5, 40, 64, 135, 193, 320])
def test_small_difference(ctx, n, precision):
    p = from_rows(n, [[(0, 0), (1, 0)], [(0, 0), (1, 0)]])
    eye = np.eye(n)
    A = chidg_matrix(p, ctx)
    A.store(np.stack([eye, eye, eye, 2 * eye]).reshape(-1))
    M = precon_ILU0(precision).init(A)
    M.update(A)
    r = np.random.default_rng(n)
    k = 8
    V = np.stack([np.concatenate([1 + 1e-9 * r.uniform(0.5, 1.5, n) * r.choice([-1, 1], n), np.full(n, 2.0)])
                  for _ in range(k)])
    ref = np.concatenate([V[:, :n] - 1, np.ones((k, n))], axis=1)
    for v, w in zip(V[:2], ref):
        assert np.all(np.abs(M.apply(A, v) - w) <= 1e-6 * np.abs(w))
    if precision == "fp32":                   # (several vectors under BF16 storage: W, whose product takes y_0 in FP32)
        for m in (2, 4, 8):
            Z = np.empty((m, 2 * n))
            ctx._check(ctx.lib.cdg_prec_apply_multi(ctx.h, M.h, A.h, m, V.ctypes.data_as(C.c_void_p),
                                                    Z.ctypes.data_as(C.c_void_p)), "cdg_prec_apply_multi")
            assert np.all(np.abs(Z - ref[:m]) <= 1e-6 * np.abs(ref[:m])), m
    M.tear_down()
    A.release()
