"""GPU: Jacobi on the two sides of the rule that gives the stop test of a launch to
the next launch or to a block of its own (2048 blocks of 112 x 48 cells), against the
oracle as in test_gpu_steps.py: u and, where the last iteration forms it, r with the
same bits after the same number of iterations, where a limit ends the solve and where
the stop rule does, inside a launch and at its end."""
import numpy as np
import pytest

import oracle as O
import tealeaf_hip as T
from tealeaf_hip import decks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(113, 49000), (113, 49440)])
def test_jacobi_stops_match_oracle(nx, ny):
    eps = 1e-15
    for limit, rule in ((8, False), (21, False), (21, True), (50, False), (24, False), (24, True)):
        print(f"case: Jacobi {nx}x{ny}, {limit} iterations by the {'stop rule' if rule else 'limit'}", flush=True)
        # the error falls from iteration to iteration: just above iteration `limit`'s it stops there
        text = decks.reference_deck(nx, 1, solver="jacobi", max_iters=1000 if rule else limit,
                                    eps=eps if rule else 1e-15).replace(f"y_cells={nx}", f"y_cells={ny}")
        d = O.parse_deck(text)
        d.checkresult = False  # the step's own residual! would replace the solve's r
        o = O.Oracle(d, threads=8)
        o.initialise()
        ost = o.step()
        s = T.Settings.from_text(text).set(check_result=0)
        c = T.initialiseapp(s)
        st = T.step(c, s)
        assert st["iterations"] == ost["iterations"] == limit, (st, ost)
        assert st["converged"] == int(rule), st
        for f in ("u",) + (("r",) if limit % 50 == 0 else ()):
            a, b = c.interior(f), o.field(f)[2:-2, 2:-2]
            assert np.array_equal(a, b), (f, limit, np.max(np.abs(a - b)))
        c.close()
        eps = st["error"] * (1 + 1e-9)


def test_cost_grows_with_the_cells():
    """Four times the cells take at most six times as long (the stop test once took a
    time that grew with the square of the grid: seven times)."""
    ms = []
    for n in (8192, 16384):
        print(f"case: Jacobi {n}^2, time of 200 iterations", flush=True)
        s = T.Settings.from_text(decks.reference_deck(n, 1, solver="jacobi", max_iters=200))
        c = T.initialiseapp(s)
        ms.append(min(s.solver.solve(c, s, s.dtinit / s.dx ** 2, s.dtinit / s.dy ** 2)["solve_ms"] for _ in range(3)))
        c.close()
    assert ms[1] < 6 * ms[0], ms
