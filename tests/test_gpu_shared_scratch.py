"""GPU: solvers that follow one another on one context share its scratch (the second
buffers of sd, p and u) and swap it with their fields.  Each solve of a sequence that
mixes them must leave, bit for bit, what the same solve leaves on a context of its own:
u and the fields that the solver defines, halos included.  Iteration counts are odd and
even, so that every swap happens and does not; the grids take the CG held in registers
and, where that is declined, the sweeps."""
import numpy as np
import pytest

import tealeaf_hip as T
from tealeaf_hip import decks

pytestmark = pytest.mark.gpu

CG, PPCG, CHEBY, JACOBI = ("u", "u0", "p", "r", "w"), ("u", "u0", "p", "r", "sd"), ("u", "u0", "p"), ("u", "u0")
REL = dict(stop_rule=T.TL_STOP_RELATIVE, rel_tol=1e-10)
SEQUENCE = [
    ("ppcg", dict(max_iters=40, ppcg_inner_steps=10), PPCG), ("cg", dict(max_iters=9), CG),
    ("jacobi", dict(max_iters=57), JACOBI), ("ppcg", dict(max_iters=41, ppcg_inner_steps=5), PPCG),
    ("cg", dict(max_iters=10), CG), ("cheby", dict(max_iters=150), CHEBY), ("jacobi", dict(max_iters=100), JACOBI + ("r",)),
    ("cg", dict(max_iters=2000, **REL), CG), ("cg", dict(max_iters=2000, precision=T.TL_FP32_IR, **REL), ("u", "u0")),
    ("jacobi", dict(max_iters=50), JACOBI + ("r",)), ("ppcg", dict(max_iters=39, ppcg_inner_steps=3), PPCG),
    ("cheby", dict(max_iters=149), CHEBY), ("cg", dict(max_iters=11), CG),
]


def _solve(c, text, solver, kw, rho, e):
    s = T.Settings.from_text(text).set(solver=solver, **kw)
    if c is None:
        c = T.initialiseapp(s)
    c.set_field("density", rho)
    c.set_field("energy", e)
    st = s.solver.solve(c, s, s.dtinit / s.dx ** 2, s.dtinit / s.dy ** 2)
    return c, st


@pytest.mark.parametrize("polls", [0, -1], ids=["registers", "sweeps"])
@pytest.mark.parametrize("nx,ny", [(131, 77), (256, 150)])
def test_sequence_equals_fresh_contexts(nx, ny, polls):
    text = decks.reference_deck(nx, 1, presteps=8).replace(f"y_cells={nx}", f"y_cells={ny}")
    g = np.random.default_rng(nx)
    rho = np.pad(10.0 ** g.uniform(-1.0, 1.0, (ny, nx)), 2, mode="symmetric")
    shared = None
    for i, (solver, kw, fields) in enumerate(SEQUENCE):
        print(f"case: {nx}x{ny}, solve {i} of the sequence, {solver} {kw}, {polls} polls", flush=True)
        e = np.pad(g.uniform(0.1, 1.0, (ny, nx)), 2, mode="symmetric")
        shared, a = _solve(shared, text, solver, dict(kw, resident_polls=polls), rho, e)
        own, b = _solve(None, text, solver, dict(kw, resident_polls=polls), rho, e)
        for k in ("iterations", "cg_iters", "cheby_iters", "refreshes", "converged", "error", "rel_resid", "cg_form"):
            assert a[k] == b[k], (i, solver, k, a[k], b[k])
        for f in fields:
            # Jacobi copies u to u0 halo and all (Jacobi.jl:38-40), the others only the interior
            x, y = (c.interior(f) if f == "u0" else c.field(f) for c in (shared, own))
            assert np.array_equal(x, y), (i, solver, f, int((x != y).sum()))
        own.close()
    shared.close()
