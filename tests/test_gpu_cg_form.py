"""GPU: which form of the CG iterations a solve takes (stats.cg_form), on both sides
of the rules that choose it, and the restart of a solve whose register-held launch
gives up.

A wait of one poll is too short for the blocks of a launch to find one another's sums
in every iteration, so some block gives up (every block then ends by the same bound).
The solve must start again in the form that resident_polls = -1 takes and give its
bits and statistics: nothing of the abandoned run is counted, a warm start is not
evaluated twice, and the context stays with that form."""
import os

import numpy as np
import pytest

import tealeaf_hip as T
from tealeaf_hip import _lib, decks, unet

pytestmark = pytest.mark.gpu

SWEEP, RESIDENT, TWO, FUSED, PAIRS = (_lib.TL_FORM_SWEEP, _lib.TL_FORM_RESIDENT, _lib.TL_FORM_TWO,
                                      _lib.TL_FORM_FUSED, _lib.TL_FORM_PAIRS)
WEIGHTS = os.path.join(os.path.dirname(_lib.__file__), "..", "weights", "unet_warmstart.npy")
STATS = ("iterations", "refreshes", "converged", "error", "rel_resid", "init_rel_resid", "start", "warm_attempted",
         "fallback")


def _text(nx, ny, precision, dt=0.004):
    return (decks.random_rect_deck(13, n=nx, steps=1, nrect=8, precision=precision)
            .replace(f"y_cells={nx}", f"y_cells={ny}").replace("initial_timestep=0.004", f"initial_timestep={dt}"))


@pytest.mark.parametrize("precision,nx,ny,kw,form", [
    ("fp64", 2, 2, {}, RESIDENT), ("fp64", 500, 300, {}, RESIDENT), ("fp64", 500, 300, {"launch": 1}, RESIDENT),
    ("fp64", 121, 8192, {}, RESIDENT), ("fp64", 121, 8195, {}, SWEEP), ("fp64", 500, 300, {"resident_polls": -1}, SWEEP),
    ("fp64", 500, 300, {"resident_polls": -1, "launch": 1}, SWEEP),
    ("fp32_ir", 128, 255, {}, PAIRS), ("fp32_ir", 128, 256, {}, RESIDENT), ("fp32_ir", 128, 256, {"launch": 1}, FUSED),
    ("fp32_ir", 128, 256, {"resident_polls": -1}, PAIRS), ("fp32_ir", 127, 128, {}, TWO),
    ("fp32_ir", 129, 128, {}, PAIRS), ("fp32_ir", 129, 128, {"launch": 1}, PAIRS), ("fp32_ir", 183, 181, {}, RESIDENT),
    ("fp32_ir", 183, 181, {"launch": 1}, RESIDENT), ("fp32_ir", 183, 181, {"resident_polls": -1}, PAIRS),
    ("fp32_ir", 241, 8192, {}, RESIDENT), ("fp32_ir", 241, 8195, {}, PAIRS),
    ("fp32_ir", 256, 256, {"fp32_kernels": 1}, TWO), ("fp32_ir", 256, 256, {"fp32_kernels": 2}, FUSED),
    ("fp32_ir", 256, 256, {"fp32_kernels": 3}, PAIRS),
])
def test_form(precision, nx, ny, kw, form):
    print(f"case: form of {precision} {nx}x{ny} {kw}", flush=True)
    s = T.Settings.from_text(_text(nx, ny, precision, 1e-7 if nx * ny > 400000 else 0.004)).set(**kw)
    c = T.initialiseapp(s)
    st = T.step(c, s)
    c.close()
    assert st["cg_form"] == form, st


@pytest.mark.parametrize("solver", ["cheby", "ppcg", "jacobi"])
def test_other_solvers_have_none(solver):
    s = T.Settings.from_text(decks.reference_deck(64, 1, solver=solver, max_iters=50))
    c = T.initialiseapp(s)
    assert T.step(c, s)["cg_form"] == 0
    c.close()


RESTARTS = [("fp64", 500, 300), ("fp64", 700, 900), ("fp32_ir", 256, 256), ("fp32_ir", 183, 181),
            ("fp32_ir", 1023, 900)]


# the learned start on grids that the network takes (edges that are multiples of 4)
@pytest.mark.parametrize("precision,nx,ny,warm", [r + ("none",) for r in RESTARTS] +
                         [r + ("learned",) for r in RESTARTS if r[1] % 4 == 0 and r[2] % 4 == 0])
def test_restart_gives_what_the_declined_form_gives(precision, nx, ny, warm):
    out = []
    for polls in (1, -1):
        print(f"case: {precision} {nx}x{ny}, warm start {warm}, {polls} polls", flush=True)
        s = T.Settings.from_text(_text(nx, ny, precision)).set(
            resident_polls=polls, warm_start=T.TL_WARM_LEARNED if warm == "learned" else T.TL_WARM_NONE)
        c = T.initialiseapp(s)
        if warm == "learned":
            unet.load_weights(c, WEIGHTS)
        rows, forms = [], []
        for t in range(3):
            st = T.step(c, s)
            rows.append([st[k] for k in STATS])
            forms.append(st["cg_form"])
        out.append((rows, [c.field(f) for f in ("u", "r", "p", "w", "energy")], forms))
        c.close()
    (ra, fa, a), (rb, fb, b) = out
    assert b == [SWEEP if precision == "fp64" else PAIRS] * 3, b
    assert a == [b[0] + _lib.TL_FORM_RESTARTED, b[0], b[0]], a  # later solves take that form at once
    assert ra == rb
    for x, y in zip(fa, fb):
        assert np.array_equal(x, y)
