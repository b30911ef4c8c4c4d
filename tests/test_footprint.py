"""The server's estimate of a request's device memory (host code): it holds the Krylov basis and the step's own
workspace, a triangle of nkrylov (nkrylov + 1) / 2 values among it, for every right-hand side and for the nested
solver."""
import ctypes as C

import pytest

from chidg_amd import _lib
from chidg_amd.linsolve import fgmres
from chidg_amd.serve import Request


def footprint(nrhs=1, **kw):
    r, p, b = Request(4, 4, 4, 1, seed_A=1, nrhs=nrhs).c(), fgmres(**kw).params(), C.c_int64()
    assert _lib.load().cdg_server_footprint(C.byref(r), C.byref(p), C.byref(b)) == 0
    return b.value


@pytest.mark.parametrize("m", [30, 2000])
def test_holds_basis_and_triangle(m):
    vec = 8 * 64 * 40
    lane = 2 * m * vec + 8 * m * (m + 1) // 2
    kw = dict(nkrylov=m, inner_fgmres=False)
    assert footprint(8, **kw) - footprint(1, **kw) >= 7 * lane
    nested = dict(nkrylov=m, inner_fgmres=True)
    inner = footprint(1, **nested, inner_nkrylov=m) - footprint(1, **kw)
    assert inner >= lane
