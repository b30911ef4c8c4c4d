"""The tuner where the sweep is the apply: it reports the time of the launch that the next apply makes, chooses
nothing, and no storage of the column-slice launches is held; choosing 'folded' or 'dataflow' takes it then."""
import time

import numpy as np
import pytest
import torch

import pyoracle as po
from chidg_amd.linsolve import Context, chidg_matrix, precon_ILU0
from helpers import synthetic_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("schedule,precision", [("auto", "fp64"), ("auto", "fp32"), ("levels", "fp64"), ("levels", "bf16"),
                                                ("rowslice", "fp32"), ("rowslice", "bf16")])
def test_tune_under_the_sweep(schedule, precision):
    ctx = Context(0)
    p, blocks = synthetic_system(6, 6, 5, 1, seed=7)
    A = chidg_matrix(p, ctx)
    A.store(blocks)
    before = ctx.mem_used()
    M = precon_ILU0(precision, schedule=schedule).init(A)
    M.update(A)
    shape, used = M.launch_shape(), ctx.mem_used()
    v = torch.from_numpy(po.fill_vector(p.vec_len, 5)).cuda()
    z = torch.empty_like(v)
    ref = M.apply(A, v).clone()
    M.tune(A, reps=1)
    tuned = M.tune(A, reps=20)
    assert M.launch_shape() == shape and ctx.mem_used() == used
    torch.cuda.synchronize()
    t = min(_timed(M, A, v, z) for _ in range(5))
    assert 0.5 * t < tuned < 2 * t
    assert torch.equal(M.apply(A, v), ref)
    if precision == "fp64":
        slices = 3 * 8 * shape["slices"] * p.vec_len
        M.set_schedule("folded")
        assert ctx.mem_used() - used >= slices
        y = M.apply(A, v)
        assert float(torch.linalg.norm(y - ref) / torch.linalg.norm(ref)) < 1e-13
        M.set_schedule("dataflow")
        y = M.apply(A, v)
        assert float(torch.linalg.norm(y - ref) / torch.linalg.norm(ref)) < 1e-13
    M.tear_down()
    assert ctx.mem_used() == before
    A.release()
    ctx.close()


def _timed(M, A, v, z, reps=20):
    torch.cuda.synchronize()
    t = time.perf_counter()
    for _ in range(reps):
        M.apply_async(A, v, z, order=False)
    torch.cuda.synchronize()
    return (time.perf_counter() - t) / reps
