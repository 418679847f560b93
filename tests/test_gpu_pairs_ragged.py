"""GPU: pairs of FP32 CG iterations on grids whose width is not a multiple of the
4 columns a lane owns (the automatic choice from 16384 cells on), in the
conventions of test_gpu_pairs.py: every step meets the FP64 true residual of
1e-10 and agrees with the oracle's FP64 solution within 1e-9 in every
field-summary quantity, and the iterations lie within 5% of the two-kernel
form's, plus the null step that each refresh may add (a pair that reaches a
refresh with its first step counts its second, a null step, as an iteration).  Widths leave 1, 2 and 3 columns of a last vector, alone in a tile's
strip and beside a full one; coefficient 2 exchanges the roles of small and
large densities."""
import numpy as np
import pytest

import oracle as O
import tealeaf_hip as T
from tealeaf_hip import _lib, decks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("coefficient", [1, 2])
@pytest.mark.parametrize("nx,ny", [(3, 5500), (130, 127), (241, 70), (243, 71), (482, 34), (1021, 17)])
def test_ragged_pairs_match_oracle(nx, ny, coefficient):
    print(f"case: ragged FP32 CG pairs {nx}x{ny}, coefficient {coefficient}", flush=True)
    text = (decks.random_rect_deck(17, n=nx, steps=1, nrect=8, precision="fp32_ir")
            .replace(f"y_cells={nx}", f"y_cells={ny}").replace("coefficient=1", f"coefficient={coefficient}"))
    d = O.parse_deck(text)
    d.stop_rule, d.rel_tol, d.maxiters = O.STOP_RELATIVE, 1e-12, 200000
    o = O.Oracle(d, threads=8)
    o.initialise()
    osum = o.run(1)[0]
    iters, refreshes = {}, {}
    for form in (_lib.TL_FP32_KERNELS_AUTO, _lib.TL_FP32_KERNELS_TWO):
        s = T.Settings.from_text(text).set(fp32_kernels=form)
        c = T.initialiseapp(s)
        summ, st = T.diffuse(c, s, 1)
        halo = c.field("u")
        c.close()
        assert st[0]["converged"] == 1 and st[0]["rel_resid"] <= 1e-10, (form, st[0])
        assert np.max(np.abs(summ[0] - osum[0]) / np.abs(osum[0])) < 1e-9, (form, summ[0], osum[0])
        assert np.array_equal(halo[2:-2, 1], halo[2:-2, 2]) and np.array_equal(halo[2:-2, -2], halo[2:-2, -3])
        iters[form], refreshes[form] = st[0]["iterations"], st[0]["refreshes"]
    a, b = iters[_lib.TL_FP32_KERNELS_AUTO], iters[_lib.TL_FP32_KERNELS_TWO]
    assert a % 2 == 0  # the pairs ran
    assert abs(a - b) <= max(6, 0.05 * b) + refreshes[_lib.TL_FP32_KERNELS_AUTO], (iters, refreshes)


@pytest.mark.parametrize("nx,ny,form", [(130, 127, "AUTO"), (128, 96, "PAIRS")])
def test_iteration_limit_adds_every_update_once(nx, ny, form):
    """A limit ends the solve inside a pair (9) or after one (10) with the partial
    correction kept.  Without a refresh (ir_delta far below what ten iterations
    reach) the pairs and the two-kernel form take the same CG steps up to FP32
    rounding, about 1e-6 of the correction; an update missing or added twice
    changes it by percents."""
    text = (decks.random_rect_deck(17, n=nx, steps=1, nrect=8, precision="fp32_ir")
            .replace(f"y_cells={nx}", f"y_cells={ny}"))
    for limit in (9, 10):
        print(f"case: FP32 CG pairs {nx}x{ny} stopped after {limit} iterations", flush=True)
        u = {}
        for f in (form, "TWO"):
            s = T.Settings.from_text(text).set(fp32_kernels=getattr(_lib, f"TL_FP32_KERNELS_{f}"), max_iters=limit,
                                               ir_delta=1e-6)
            c = T.initialiseapp(s)
            st = T.step(c, s)
            assert st["iterations"] == limit and st["refreshes"] == 0, st
            u[f], u0 = c.interior("u"), c.interior("u0")
            c.close()
        assert np.linalg.norm(u[form] - u["TWO"]) <= 1e-4 * np.linalg.norm(u["TWO"] - u0)
