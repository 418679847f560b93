"""GPU: an FP32 solve whose vectors overflow leaves nothing behind that a later
solve on the same context reads.

On widths that are not a multiple of 4 the pairs of iterations store whole
vectors, the columns beside the domain included.  Where A p is infinite at the
last column, the results are NaN, there and beside it (0 times infinity).  The
densities and energies are drawn so that this happens in a later pair than the
first: a few light cells in the last column, a step of the energy some columns
before it, and noise; the scale runs over three decades, in which the overflow
moves from no iteration to the first.  Whatever each of these solves ends in, the
ordinary solve that follows must meet its tolerance and give the bits that it gave
before."""
import numpy as np
import pytest

import tealeaf_hip as T
from tealeaf_hip import _lib, decks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(130, 127), (129, 128), (131, 126)])
def test_ordinary_solve_after_an_overflow(nx, ny):
    text = (decks.random_rect_deck(17, n=nx, steps=1, nrect=8, precision="fp32_ir")
            .replace(f"y_cells={nx}", f"y_cells={ny}"))
    s = T.Settings.from_text(text)
    c = T.initialiseapp(s)
    rx, ry = s.dtinit / s.dx ** 2, s.dtinit / s.dy ** 2
    rho, e = c.field("density"), c.field("energy")
    st = s.solver.solve(c, s, rx, ry)
    want = c.field("u")
    assert st["converged"] == 1
    broke = 0
    for seed in range(10):
        print(f"case: FP32 CG pairs {nx}x{ny}, overflowing fields of seed {seed}", flush=True)
        g = np.random.default_rng(seed)
        light = np.full((ny, nx), 10.0 ** g.uniform(0, 2))
        for _ in range(g.integers(1, 6)):
            light[g.integers(0, ny), nx - 1] = 10.0 ** g.uniform(-3, -1)
        step = np.zeros((ny, nx))
        step[:, :nx - g.integers(1, 12)] = 1.0
        step += 10.0 ** g.uniform(-6, -1) * g.uniform(0, 1, (ny, nx))
        light, step = np.pad(light, 2, mode="symmetric"), np.pad(step, 2, mode="symmetric")
        for k in np.arange(34.9, 38.0, 0.2):
            c.set_field("density", light)
            c.set_field("energy", step * 10.0 ** k / light)
            try:
                s.set(max_iters=40).solver.solve(c, s, rx, ry)
            except T.TeaLeafError as err:
                assert err.code == _lib.TL_E_BREAKDOWN, err
                broke += 1
            c.set_field("density", rho)
            c.set_field("energy", e)
            st = s.set(max_iters=100000).solver.solve(c, s, rx, ry)
            assert st["converged"] == 1 and st["rel_resid"] <= 1e-10, (seed, k, st)
            assert np.array_equal(c.field("u"), want), (seed, k)
    assert broke > 0
    c.close()
