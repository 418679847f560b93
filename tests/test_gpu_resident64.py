"""GPU: the FP64 CG held in registers over many iterations, against the oracle's
CG in the conventions of test_gpu_sweep64.py: every field-summary quantity within
1e-10, u and p within 1e-9 of u's scale, iterations within max(3, 2%).  The grids
lie at the edges of its tiles (120 columns by 2 or 4 rows, one or several waves
and blocks) and of the rule that takes it: 2048 tiles of 2 rows, then of 4, 1024
of 12, then of 16, then one sweep per iteration, which is also run at each of these sizes (it is the form
that launches timed one by one take).  A launch holds up to 256 iterations; one
grid needs several."""
import numpy as np
import pytest

import oracle as O
import tealeaf_hip as T
from tealeaf_hip import _lib, decks

pytestmark = pytest.mark.gpu

SWEEPS = (1 << 0) | (1 << 1)  # TL_K_CG_W64, TL_K_CG_UR64

SMALL = [(2, 2), (119, 15), (120, 16), (121, 17), (122, 35), (241, 34), (700, 3)]
EDGES = [(121, 2047), (121, 2050), (1081, 410), (121, 4095), (121, 4098), (121, 6144), (121, 6147), (121, 8192),
         (121, 8195), (1500, 1100)]


def _check(nx, ny, coefficient, max_iters, sweeps):
    text = (decks.reference_deck(nx, 1, max_iters=max_iters).replace(f"y_cells={nx}", f"y_cells={ny}")
            .replace("coefficient=1", f"coefficient={coefficient}"))
    o = O.Oracle(O.parse_deck(text), threads=8)
    o.initialise()
    osum, ost = o.run(1)
    s = T.Settings.from_text(text)
    c = T.initialiseapp(s)
    if sweeps:
        _lib.check(_lib.load().tl_profile_begin(c._ctx, SWEEPS, 1), c._ctx, "tl_profile_begin")
    gsum, gst = T.diffuse(c, s, 1)
    assert np.max(np.abs(gsum[0] - osum[0]) / np.abs(osum[0])) < 1e-10, (gsum[0], osum[0])
    scale = np.max(np.abs(o.field("u")))
    for f in ("u", "p"):
        assert np.max(np.abs(c.field(f) - o.field(f))) <= 1e-9 * scale, f
    c.close()
    return gst[0], ost[0]


@pytest.mark.parametrize("sweeps", [False, True], ids=["resident", "sweeps"])
@pytest.mark.parametrize("nx,ny", SMALL + [(500, 300)])
def test_solve_matches_oracle(nx, ny, sweeps):
    for coefficient in (1, 2):
        print(f"case: FP64 CG {nx}x{ny}, coefficient {coefficient}, {'sweeps' if sweeps else 'automatic'}", flush=True)
        g, o = _check(nx, ny, coefficient, 10000, sweeps)
        assert g["converged"] == 1
        assert abs(g["iterations"] - o["iterations"]) <= max(3, o["iterations"] // 50), (g, o)


@pytest.mark.parametrize("sweeps", [False, True], ids=["resident", "sweeps"])
@pytest.mark.parametrize("nx,ny", SMALL + EDGES)
def test_iteration_limit_matches_oracle(nx, ny, sweeps):
    for limit in (1, 2, 5, 40):
        print(f"case: FP64 CG {nx}x{ny} stopped after {limit}, {'sweeps' if sweeps else 'automatic'}", flush=True)
        g, o = _check(nx, ny, 1, limit, sweeps)
        assert g["iterations"] == o["iterations"] <= limit


def test_graph_batches_of_the_sweeps_bit_identical_to_stream():
    out = []
    for launch in (T.TL_LAUNCH_STREAM, T.TL_LAUNCH_GRAPH):
        print(f"case: FP64 CG sweeps 256^2, 2 steps, launch {launch}", flush=True)
        s = T.Settings.from_text(decks.random_rect_deck(3, n=256, steps=2)).set(launch=launch)
        c = T.initialiseapp(s)
        _lib.check(_lib.load().tl_profile_begin(c._ctx, SWEEPS, 1), c._ctx, "tl_profile_begin")
        summ, st = T.diffuse(c, s, 2)
        out.append((summ, [x["iterations"] for x in st], c.field("u"), c.field("p"), c.field("r")))
        c.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    assert min(out[0][1]) > 64  # the graph run replays
