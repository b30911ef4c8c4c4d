"""BF16-stored ILU(0): the FP32 roundings behind its factor.  A block that is the identity but for 16 rows and columns
(one panel of the block inverse) is inverted by that panel's 16 pivot steps alone: what they leave is repeated here
in FP32, step by step, and every stored BF16 value must be the same.  (A value that FP32 rounds the other way would
land on another BF16 value once in 20000.)  The products and sums are done in FP64 and rounded once, as a fused
multiply-add rounds; a quotient that a reciprocal's Newton step misses by an ulp is one in 4e6."""
import numpy as np
import pytest

from chidg_amd.linsolve import Context, chidg_matrix, precon_ILU0
from chidg_amd.pattern import from_rows

f32 = np.float32


def bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return ((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32).view(np.float32)


def steps(a):
    """The inverses of (count, w, w) FP32 blocks by unblocked Gauss-Jordan on diagonal pivots."""
    a = a.astype(f32).copy()
    w = a.shape[1]
    for j in range(w):
        rinv = f32(1) / a[:, j, j]
        sv = a[:, j, :] * rinv[:, None]
        sv[:, j] = rinv
        cc = a[:, :, j].copy()
        upd = (a.astype(np.float64) - cc[:, :, None].astype(np.float64) * sv[:, None, :]).astype(f32)
        upd[:, :, j] = -cc * rinv[:, None]
        upd[:, j, :] = sv
        a = upd
    eye = np.eye(w, dtype=f32)
    return (a - eye) + eye          # the panel keeps its values with the identity taken off


def inputs(count, w, seed):
    r = np.random.default_rng(seed)
    return (r.standard_normal((count, w, w)) * 0.3 + 2 * np.eye(w)).astype(f32)


def test_steps_invert():
    a = inputs(50, 16, 1)
    assert np.abs(steps(a) @ a - np.eye(16)).max() < 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("n,k0,count", [(16, 0, 4000), (13, 0, 4000), (5, 0, 4000), (17, 0, 2000), (48, 32, 1500),
                                        (49, 16, 1000), (96, 64, 500), (97, 96, 200), (135, 48, 400), (144, 128, 300),
                                        (193, 16, 150), (256, 64, 100), (320, 0, 100), (320, 304, 100)])
def test_one_panel(n, k0, count):
    w = min(16, n - k0)
    a = inputs(count, w, n + k0)
    blocks = np.tile(np.eye(n), (count, 1, 1))
    blocks[:, k0:k0 + w, k0:k0 + w] = a
    ctx = Context(0)
    A = chidg_matrix(from_rows(n, [[(i, 0)] for i in range(count)]), ctx)
    A.store(np.ascontiguousarray(blocks.transpose(0, 2, 1)).reshape(-1))
    M = precon_ILU0("bf16").init(A)
    M.update(A)
    D = np.asarray(M.factors(A)[1]).reshape(count, n, n).transpose(0, 2, 1).astype(f32)
    M.tear_down()
    A.release()
    ctx.close()
    ref = np.tile(np.eye(n, dtype=f32), (count, 1, 1))
    ref[:, k0:k0 + w, k0:k0 + w] = bf16(steps(a))
    assert np.count_nonzero(D != ref) == 0
