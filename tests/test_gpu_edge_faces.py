"""GPU: several Chebyshev or PPCG steps per sweep against one per sweep, bit for
bit, where the density varies up to the domain's edges, so that the face
coefficients beside the last column differ from column to column (the decks of
the other tests have one density there).  Widths: a whole number of waves (128
columns), one vector more, odd ones, and grids of few tiles and of many."""
import numpy as np
import pytest

import tealeaf_hip as T
from tealeaf_hip import _lib, decks

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(128, 40), (130, 40), (131, 41), (256, 70), (1792, 780), (1794, 771), (1803, 771)])
@pytest.mark.parametrize("solver,key,off", [("cheby", "cheby_pairs", _lib.TL_CHEBY_PAIRS_OFF),
                                            ("ppcg", "ppcg_pairs", _lib.TL_PPCG_PAIRS_OFF)])
def test_several_steps_bit_identical_with_varying_density(nx, ny, solver, key, off):
    print(f"case: {solver} several steps per sweep vs one, {nx}x{ny}, random density", flush=True)
    text = (decks.reference_deck(nx, 1, solver=solver, presteps=8, max_iters=300)
            .replace(f"y_cells={nx}", f"y_cells={ny}"))
    g = np.random.default_rng(nx * 1000 + ny)
    rho = np.pad(10.0 ** g.uniform(-1.0, 1.0, (ny, nx)), 2, mode="symmetric")
    e = np.pad(g.uniform(0.1, 1.0, (ny, nx)), 2, mode="symmetric")
    out = []
    for pairs in (0, off):
        s = T.Settings.from_text(text).set(**{key: pairs})
        c = T.initialiseapp(s)
        c.set_field("density", rho)
        c.set_field("energy", e)
        st = T.step(c, s)
        out.append(({f: c.field(f) for f in ("u", "r", "sd", "p", "w", "u0")}, st))
        c.close()
    (fa, a), (fb, b) = out
    for k in ("iterations", "cg_iters", "cheby_iters", "error", "eigmin", "eigmax", "converged"):
        assert a[k] == b[k], (k, a[k], b[k])
    assert a["cheby_iters"] > 2, a
    for f in fa:
        d = fa[f] != fb[f]
        assert not d.any(), (f, int(d.sum()), np.max(np.abs(fa[f] - fb[f])))
