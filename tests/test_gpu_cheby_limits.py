"""GPU: how many Chebyshev iterations a launch takes near the iterations with a residual
norm and near the iteration limit: for limits that end 0 to 21 iterations after the
switch, and for a solve whose estimate is thousands of iterations away, so that most
launches lie far from the next norm, every field and statistic equals one iteration per
launch, bit for bit."""
import numpy as np
import pytest

import tealeaf_hip as T
from tealeaf_hip import _lib, decks

pytestmark = pytest.mark.gpu


def _run(text, pairs):
    s = T.Settings.from_text(text).set(cheby_pairs=pairs)
    c = T.initialiseapp(s)
    st = s.solver.solve(c, s, s.dtinit / s.dx ** 2, s.dtinit / s.dy ** 2)
    out = {f: c.field(f) for f in ("u", "r", "p")}
    c.close()
    return {k: st[k] for k in ("iterations", "cg_iters", "cheby_iters", "est_iters", "error", "converged")}, out


def _same(text):
    (a, fa), (b, fb) = _run(text, 0), _run(text, _lib.TL_CHEBY_PAIRS_OFF)
    assert a == b, (a, b)
    for f in fa:
        assert np.array_equal(fa[f], fb[f]), f
    return a


def test_limits_near_a_norm():
    for limit in range(30, 52):
        print(f"case: Chebyshev 64x40, limit {limit}", flush=True)
        st = _same(decks.reference_deck(64, 1, solver="cheby", max_iters=limit, eps=1e-300, presteps=30)
                   .replace("y_cells=64", "y_cells=40"))
        assert st["iterations"] == max(limit, 31)  # 30 CG steps, and the first Chebyshev step follows the switch


def test_estimate_far_away():
    for limit in (1999, 4000):
        print(f"case: Chebyshev 64^2, long timestep, limit {limit}", flush=True)
        st = _same(decks.reference_deck(64, 1, solver="cheby", max_iters=limit, eps=1e-300, presteps=30)
                   .replace("initial_timestep=0.004", "initial_timestep=100.0"))
        assert st["est_iters"] > 2000 and st["cheby_iters"] > 1000, st
