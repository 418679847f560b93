"""GPU: the automatic FP32 form on grids whose width is not a multiple of 4 takes
the same kernels with stream launches and with TL_LAUNCH_GRAPH, so both give the
same bits: fields, iterations and residuals of every timestep.  Sizes lie on both
sides of the two rules that choose the form (two kernels, pairs of iterations,
many iterations per launch) and beyond the last."""
import numpy as np
import pytest

import tealeaf_hip as T
from tealeaf_hip import decks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,dt", [(127, 128, 0.004), (130, 127, 0.004), (182, 180, 0.004), (183, 181, 0.004),
                                      (250, 201, 0.004), (241, 16395, 1e-7)])
def test_ragged_automatic_form_same_bits_in_both_modes(nx, ny, dt):
    text = (decks.random_rect_deck(11, n=nx, steps=2, nrect=8, precision="fp32_ir")
            .replace(f"y_cells={nx}", f"y_cells={ny}").replace("initial_timestep=0.004", f"initial_timestep={dt}"))
    out = []
    for launch in (T.TL_LAUNCH_STREAM, T.TL_LAUNCH_GRAPH):
        print(f"case: automatic FP32 form {nx}x{ny}, launch mode {launch}", flush=True)
        s = T.Settings.from_text(text).set(launch=launch)
        c = T.initialiseapp(s)
        summ, st = T.diffuse(c, s, 2)
        out.append([summ, c.field("u"), c.field("energy"),
                    [(x["iterations"], x["refreshes"], x["rel_resid"], x["converged"]) for x in st]])
        c.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert all(x[3] == 1 for x in out[0][3])
