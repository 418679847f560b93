"""GPU: the FP64 CG's one sweep per iteration on grids that the automatic choice holds
in registers (resident_polls = -1 declines that; the solve's statistics name the form).

The grids of test_gpu_sweep64.py, against the oracle in its conventions: every
field-summary quantity within 1e-10, u and p within 1e-9 of u's scale, iterations
within max(3, 2%), and limits of 1, 2 and 3 iterations.  The FP64 cases of
test_gpu_graph.py, whose replays these sweeps are: reference and relative stop rule, a
halo of 4, an odd width; fields and statistics of every timestep with the same bits
as with stream launches."""
import numpy as np
import pytest

import oracle as O
import tealeaf_hip as T
from tealeaf_hip import _lib, decks

pytestmark = pytest.mark.gpu

GRIDS = [(2, 3), (119, 4), (120, 5), (121, 7), (122, 33), (241, 130), (601, 203)]
FIELDS = ("density", "energy", "u", "u0", "p", "r", "w", "kx", "ky")
STATS = ("iterations", "cg_iters", "refreshes", "converged", "error", "rel_resid", "init_rel_resid")
REL = "stop_rule=relative\nrel_tol=1e-10\n"


def _both(nx, ny, coefficient, max_iters):
    text = (decks.reference_deck(nx, 1, max_iters=max_iters).replace(f"y_cells={nx}", f"y_cells={ny}")
            .replace("coefficient=1", f"coefficient={coefficient}"))
    o = O.Oracle(O.parse_deck(text), threads=4)
    o.initialise()
    osum, ost = o.run(1)
    s = T.Settings.from_text(text).set(resident_polls=-1)
    c = T.initialiseapp(s)
    gsum, gst = T.diffuse(c, s, 1)
    assert gst[0]["cg_form"] == _lib.TL_FORM_SWEEP
    assert np.max(np.abs(gsum[0] - osum[0]) / np.abs(osum[0])) < 1e-10, (gsum[0], osum[0])
    scale = np.max(np.abs(o.field("u")))
    for f in ("u", "p"):
        assert np.max(np.abs(c.field(f) - o.field(f))) <= 1e-9 * scale, f
    c.close()
    return gst[0], ost[0]


@pytest.mark.parametrize("coefficient", [1, 2])
@pytest.mark.parametrize("nx,ny", GRIDS)
def test_solve_matches_oracle(nx, ny, coefficient):
    print(f"case: FP64 CG sweeps {nx}x{ny}, coefficient {coefficient}", flush=True)
    g, o = _both(nx, ny, coefficient, 10000)
    assert g["converged"] == 1
    assert abs(g["iterations"] - o["iterations"]) <= max(3, o["iterations"] // 50), (g, o)


@pytest.mark.parametrize("nx,ny", GRIDS)
def test_iteration_limit_matches_oracle(nx, ny):
    for limit in (1, 2, 3):
        print(f"case: FP64 CG sweeps {nx}x{ny} stopped after {limit} iterations", flush=True)
        g, o = _both(nx, ny, 1, limit)
        assert g["iterations"] == o["iterations"] <= limit  # fewer: the smallest grid's deck is uniform


@pytest.mark.parametrize("text,steps,replays", [
    (decks.random_rect_deck(3, n=256, steps=3), 3, True),
    (decks.reference_deck(128, 2, max_iters=700), 2, True),
    (decks.reference_deck(67, 2, extra=REL).replace("y_cells=67", "y_cells=3").replace("halo_depth=2", "halo_depth=4"),
     2, False),
    (decks.random_rect_deck(5, n=203, steps=2, nrect=8).replace("y_cells=203", "y_cells=331"), 2, True),
], ids=["relative 256^2", "reference rule 128^2", "halo 4, 67x3", "odd width 203x331"])
def test_graph_replays_bit_identical_to_stream(text, steps, replays):
    out = []
    for launch in (T.TL_LAUNCH_STREAM, T.TL_LAUNCH_GRAPH):
        print(f"case: FP64 CG sweeps, launch mode {launch}", flush=True)
        s = T.Settings.from_text(text).set(launch=launch, resident_polls=-1)
        c = T.initialiseapp(s)
        rows = []
        for _ in range(steps):
            st = T.step(c, s)
            assert st["cg_form"] == _lib.TL_FORM_SWEEP
            assert st["iterations"] > (64 if replays else 5)
            rows.append((T.fieldsummary(c), [st[k] for k in STATS], [c.field(f) for f in FIELDS]))
        c.close()
        out.append(rows)
    for a, b in zip(*out):
        assert np.array_equal(a[0], b[0]) and a[1] == b[1], (a[:2], b[:2])
        for x, y in zip(a[2], b[2]):
            assert np.array_equal(x, y)
