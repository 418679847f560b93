"""GPU: mixed-precision solves of fields so small that the FP32 residual underflows
end, in every form of the inner CG and for every launch mode.

The FP64 residual, which decides, then stays above the tolerance while sums over
the FP32 residual are zero.  A form that took its stop test from those sums would
ask for the same refresh again without an iteration between, which no iteration
limit ends.  What such a solve gives is convergence on the true residual, a
breakdown (p A p = 0) or the iteration limit."""
import pytest

import tealeaf_hip as T
from tealeaf_hip import _lib, decks

pytestmark = pytest.mark.gpu

FORMS = [("AUTO", 0), ("AUTO", 1), ("FUSED", 0), ("FUSED", 1), ("PAIRS", 0), ("TWO", 0), ("TWO", 1)]


@pytest.mark.parametrize("form,launch", FORMS)
@pytest.mark.parametrize("nx,ny", [(256, 160), (100, 80)])
def test_solve_ends(nx, ny, form, launch):
    text = (decks.random_rect_deck(7, n=nx, steps=1, nrect=8, precision="fp32_ir", max_iters=3000)
            .replace(f"y_cells={nx}", f"y_cells={ny}"))
    for scale in (1e-20, 1e-30, 1e-34, 1e-36, 1e-38, 1e-42):
        print(f"case: FP32 CG {nx}x{ny}, form {form}, launch {launch}, energies times {scale}", flush=True)
        s = T.Settings.from_text(text).set(fp32_kernels=getattr(_lib, f"TL_FP32_KERNELS_{form}"), launch=launch)
        c = T.initialiseapp(s)
        c.set_field("energy", c.field("energy") * scale)
        try:
            st = s.solver.solve(c, s, s.dtinit / s.dx ** 2, s.dtinit / s.dy ** 2)
            assert st["iterations"] <= 3000
            assert st["rel_resid"] <= 1e-10 if st["converged"] else st["iterations"] == 3000, st
        except T.TeaLeafError as err:
            assert err.code == _lib.TL_E_BREAKDOWN and scale < 1e-25, err
        c.close()
