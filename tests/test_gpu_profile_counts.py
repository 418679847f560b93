"""GPU: the kernels that Chebyshev's and PPCG's CG phase launches are timed under
their ids (TL_K_CG_W64, TL_K_CG_UR64, TL_K_CG_P64): one sample per CG iteration,
and for W64 and P64 one per outer PPCG iteration as well."""
import ctypes as C

import pytest

import tealeaf_hip as T
from tealeaf_hip import _lib, decks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", ["cheby", "ppcg"])
def test_cg_phase_is_timed(solver):
    print(f"case: {solver} 200^2, timed kernels of the CG phase", flush=True)
    s = T.Settings.from_text(decks.reference_deck(200, 1, solver=solver, presteps=8, max_iters=300))
    c = T.initialiseapp(s)
    L = _lib.load()
    ids = (_lib.TL_K_CG_W64, _lib.TL_K_CG_UR64, _lib.TL_K_CG_P64)
    _lib.check(L.tl_profile_begin(c._ctx, sum(1 << k for k in ids), 1), c._ctx, "tl_profile_begin")
    st = T.step(c, s)
    n = C.c_int()
    got = []
    for k in ids:
        _lib.check(L.tl_profile_read(c._ctx, k, None, 0, C.byref(n)), c._ctx, "tl_profile_read")
        got.append(n.value)
    c.close()
    # launches past the stop exit at once and are timed as well
    outer = st["cheby_iters"] if solver == "ppcg" else 0
    assert got[0] >= st["cg_iters"] + outer and got[2] >= st["cg_iters"] + outer, (got, st)
    assert got[1] >= st["cg_iters"], (got, st)
