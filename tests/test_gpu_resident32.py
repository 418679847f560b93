"""GPU: the FP32 inner CG held in registers over many iterations (the automatic
choice from 32768 cells up to 1024 tiles of 240 columns by 16 rows), in the
conventions of test_gpu_pairs.py: every step meets the FP64 true residual of
1e-10, agrees with the oracle's FP64 solution within 1e-9 in every field-summary
quantity, and takes as many iterations as the two-kernel form within 5%.  Widths
lie around one and two tiles and leave 1, 2 and 3 columns of a last vector;
heights leave a remainder of the rows of a tile.  The long grids lie at the edges of
the rule (2048 tiles of 2 rows, of 4, 1024 of 12, of 16, and beyond, where the pairs run,
whose refreshes may add a counted null step each, as in test_gpu_pairs_ragged.py),
with a short timestep that keeps their solves to some tens of iterations."""
import numpy as np
import pytest

import oracle as O
import tealeaf_hip as T
from tealeaf_hip import _lib, decks

pytestmark = pytest.mark.gpu

GRIDS = [(240, 137, 0.004), (241, 140, 0.004), (242, 137, 0.004), (243, 139, 0.004), (479, 71, 0.004),
         (482, 69, 0.004), (1100, 31, 0.004),
         (241, 2047, 4e-6), (241, 2050, 4e-6), (241, 4095, 1e-6), (241, 4098, 1e-6),
         (241, 6144, 4e-7), (241, 6147, 4e-7), (241, 8192, 2e-7), (241, 8195, 2e-7), (2047, 1533, 4e-6)]


@pytest.mark.parametrize("coefficient", [1, 2])
@pytest.mark.parametrize("nx,ny,dt", GRIDS)
def test_resident_matches_oracle(nx, ny, dt, coefficient):
    print(f"case: FP32 CG in registers {nx}x{ny}, coefficient {coefficient}", flush=True)
    text = (decks.random_rect_deck(19, n=nx, steps=2, nrect=8, precision="fp32_ir")
            .replace(f"y_cells={nx}", f"y_cells={ny}").replace("coefficient=1", f"coefficient={coefficient}")
            .replace("initial_timestep=0.004", f"initial_timestep={dt}"))
    d = O.parse_deck(text)
    d.stop_rule, d.rel_tol, d.maxiters = O.STOP_RELATIVE, 1e-12, 200000
    o = O.Oracle(d, threads=8)
    o.initialise()
    osum = o.run(2)[0]
    iters = {}
    pairs = -(-nx // 240) * -(-ny // 16) > 1024
    for form in (_lib.TL_FP32_KERNELS_TWO, _lib.TL_FP32_KERNELS_AUTO):
        s = T.Settings.from_text(text).set(fp32_kernels=form)
        c = T.initialiseapp(s)
        summ, st = T.diffuse(c, s, 2)
        c.close()
        for t in range(2):
            assert st[t]["converged"] == 1 and st[t]["rel_resid"] <= 1e-10, (form, t, st[t])
            assert np.max(np.abs(summ[t] - osum[t]) / np.abs(osum[t])) < 1e-9, (form, t, summ[t], osum[t])
        iters[form] = [x["iterations"] for x in st]
        null = [x["refreshes"] if pairs else 0 for x in st]
    for a, b, n in zip(iters[_lib.TL_FP32_KERNELS_AUTO], iters[_lib.TL_FP32_KERNELS_TWO], null):
        assert abs(a - b) <= max(6, 0.05 * b) + n, iters


def test_iteration_limit():
    """A limit of 9 or 10 iterations ends the solve there, unconverged, with the
    partial correction kept: the true residual is below the starting one."""
    text = decks.random_rect_deck(5, n=256, steps=1, nrect=8, precision="fp32_ir")
    for lim in (9, 10):
        print(f"case: FP32 CG in registers 256^2 stopped after {lim}", flush=True)
        s = T.Settings.from_text(text).set(max_iters=lim)
        c = T.initialiseapp(s)
        _, st = T.diffuse(c, s, 1)
        c.close()
        assert st[0]["iterations"] == lim and st[0]["converged"] == 0, st[0]
        assert st[0]["rel_resid"] < st[0]["init_rel_resid"], st[0]


def test_bfloat16_coefficients():
    """A density range beyond a scaled half's: the coefficients are held as
    bfloat16 (the formats and decks of test_gpu_parity.py, on a grid that is held
    in registers)."""
    print("case: FP32 CG in registers 200x180, bfloat16 coefficients", flush=True)
    text = decks.reference_deck(200, 2, extra="stop_rule=relative\nrel_tol=1e-10\nprecision=fp32_ir\n")
    text = text.replace("y_cells=200", "y_cells=180").replace("density=100.0", "density=1e5").replace("density=0.1",
                                                                                                      "density=1e-5")
    d = O.parse_deck(text)
    d.stop_rule, d.rel_tol, d.maxiters = O.STOP_RELATIVE, 1e-12, 200000
    o = O.Oracle(d, threads=8)
    o.initialise()
    osum = o.run(2)[0]
    c = T.initialiseapp(T.Settings.from_text(text))
    summ, st = T.diffuse(c, T.Settings.from_text(text), 2)
    c.close()
    for t in range(2):
        assert st[t]["coef_format"] == _lib.TL_COEF_BF16, st[t]
        assert st[t]["converged"] == 1 and st[t]["rel_resid"] <= 1e-10, (t, st[t])
        assert np.max(np.abs(summ[t] - osum[t]) / np.abs(osum[t])) < 1e-9, (t, summ[t], osum[t])
