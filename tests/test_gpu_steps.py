"""GPU: several solver steps per sweep (k_steps) on the tile shapes that the
small grids of test_gpu_two_step.py do not reach, and Jacobi's stop inside a
launch.

Chebyshev and PPCG: every field and statistic bit-identical to one step per
sweep, as there.  1003x500 takes many tiles of 64x32 cells, 1803x771 tiles of
128x64, both with an odd width and a last row of tiles that is cut.

Jacobi (760x128 has the 256 tiles of 64x24 cells that it takes at most, 760x129
more): the iteration limit is not a multiple of the steps per launch, so the
solve stops inside one and the remaining steps are repeated; u is compared with
the oracle's Jacobi after the same number of iterations, and r, which the
reference also uses as scratch, where the last iteration forms the residual
(every 50th).  Both sides round every operation alike, so u and r are equal;
the error sums differ by their order only."""
import numpy as np
import pytest

import oracle as O
import tealeaf_hip as T
from tealeaf_hip import _lib, decks

pytestmark = pytest.mark.gpu


def _deck(nx, ny, solver, **kw):
    return decks.reference_deck(nx, 1, solver=solver, **kw).replace(f"y_cells={nx}", f"y_cells={ny}")


def _run(text, key, off):
    s = T.Settings.from_text(text).set(**{key: off})
    c = T.initialiseapp(s)
    st = T.step(c, s)
    out = {f: c.field(f) for f in ("u", "r", "sd", "p", "w", "u0")}
    c.close()
    return st, out


@pytest.mark.parametrize("nx,ny", [(1003, 500), (1803, 771)])
@pytest.mark.parametrize("solver,key,inner", [("cheby", "cheby_pairs", 10), ("ppcg", "ppcg_pairs", 10),
                                              ("ppcg", "ppcg_pairs", 13)])
def test_large_tiles_bit_identical_to_single_steps(nx, ny, solver, key, inner):
    print(f"case: {solver} several steps per sweep vs one, {nx}x{ny}, {inner} inner steps", flush=True)
    text = _deck(nx, ny, solver, presteps=8, ppcg_inner_steps=inner, max_iters=1200)
    a, fa = _run(text, key, 0)
    b, fb = _run(text, key, _lib.TL_CHEBY_PAIRS_OFF)
    for k in ("iterations", "cg_iters", "cheby_iters", "est_iters", "error", "eigmin", "eigmax", "converged"):
        assert a[k] == b[k], (k, a[k], b[k])
    assert a["cheby_iters"] > 20
    for f in fa:
        assert np.array_equal(fa[f], fb[f]), f


@pytest.mark.parametrize("nx,ny", [(3, 2), (47, 20), (131, 77), (760, 128), (760, 129), (1003, 500), (1803, 771)])
def test_jacobi_iteration_limits_match_oracle(nx, ny):
    for limit in (1, 8, 21, 49, 50, 57, 107):
        print(f"case: Jacobi {nx}x{ny}, {limit} iterations", flush=True)
        text = _deck(nx, ny, "jacobi", max_iters=limit)
        d = O.parse_deck(text)
        d.checkresult = False  # the step's own residual! would replace the solve's r
        o = O.Oracle(d, threads=8)
        o.initialise()
        ost = o.step()
        s = T.Settings.from_text(text).set(check_result=0)
        c = T.initialiseapp(s)
        st = T.step(c, s)
        assert st["iterations"] == ost["iterations"], (st, ost)
        for f in ("u",) + (("r",) if st["iterations"] % 50 == 0 else ()):
            a, b = c.interior(f), o.field(f)[2:-2, 2:-2]
            assert np.array_equal(a, b), (f, limit, np.max(np.abs(a - b)))
        c.close()
