"""GPU: the FP64 CG's single-sweep iteration at the edges of its tiles, against
the oracle's CG, in the conventions of the other parity tests: every
field-summary quantity within 1e-10, u and p within 1e-9 of u's scale, and the
iterations within max(3, 2%).  Widths lie around one and two tiles of 120
columns, with odd ones and a sliver of one column; heights leave bands of four
rows with a remainder, and one grid has more tiles than one run of 16 per
XCD.  Limits of 1, 2 and 3 iterations stop the sweeps at odd and even ones (u
is updated for two at a time)."""
import numpy as np
import pytest

import oracle as O
import tealeaf_hip as T
from tealeaf_hip import decks

pytestmark = pytest.mark.gpu

GRIDS = [(2, 3), (119, 4), (120, 5), (121, 7), (122, 33), (241, 130), (601, 203)]


def _both(nx, ny, coefficient, max_iters):
    text = (decks.reference_deck(nx, 1, max_iters=max_iters).replace(f"y_cells={nx}", f"y_cells={ny}")
            .replace("coefficient=1", f"coefficient={coefficient}"))
    o = O.Oracle(O.parse_deck(text), threads=4)
    o.initialise()
    osum, ost = o.run(1)
    s = T.Settings.from_text(text)
    c = T.initialiseapp(s)
    gsum, gst = T.diffuse(c, s, 1)
    assert np.max(np.abs(gsum[0] - osum[0]) / np.abs(osum[0])) < 1e-10, (gsum[0], osum[0])
    scale = np.max(np.abs(o.field("u")))
    for f in ("u", "p"):
        assert np.max(np.abs(c.field(f) - o.field(f))) <= 1e-9 * scale, f
    c.close()
    return gst[0], ost[0]


@pytest.mark.parametrize("coefficient", [1, 2])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_solve_matches_oracle(nx, ny, coefficient):
    print(f"case: FP64 CG {nx}x{ny}, coefficient {coefficient}", flush=True)
    g, o = _both(nx, ny, coefficient, 10000)
    assert g["converged"] == 1
    assert abs(g["iterations"] - o["iterations"]) <= max(3, o["iterations"] // 50), (g, o)


@pytest.mark.parametrize("nx,ny", GRIDS)
def test_iteration_limit_matches_oracle(nx, ny):
    for limit in (1, 2, 3):
        print(f"case: FP64 CG {nx}x{ny} stopped after {limit} iterations", flush=True)
        g, o = _both(nx, ny, 1, limit)
        assert g["iterations"] == o["iterations"] <= limit  # fewer: the smallest grid's deck is uniform
