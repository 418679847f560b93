"""GPU: solves on a card that has no room for another field.

A context holds what its solvers need once it is created; scratch that a solver
would like beyond that must not be a condition of the solve.  The card is filled
until less than one field is left (1 GiB or more, for the runtime), and FP64 CG
by both rules, Jacobi and the automatic FP32 form on a width that is not a
multiple of 4 must give what they give on an empty card: the same field summary
and iterations (FP32: within the tolerance, the form may differ)."""
import ctypes as C

import numpy as np
import pytest

import tealeaf_hip as T
from tealeaf_hip import _lib, decks

pytestmark = pytest.mark.gpu

GIB = 1 << 30


class Filler:
    """Allocates all but `left` bytes of the card."""

    def __init__(self, left):
        T.load()
        self.hip = C.CDLL("libamdhip64.so.7")  # the runtime the library has loaded
        self.hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.hip.hipFree.argtypes = [C.c_void_p]
        self.hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
        self.left, self.held = left, []

    def free(self):
        f, t = C.c_size_t(), C.c_size_t()
        assert self.hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    def __enter__(self):
        for size in (16 * GIB, GIB, 64 << 20):
            while self.free() >= self.left + size:
                p = C.c_void_p()
                if self.hip.hipMalloc(C.byref(p), size) != 0:
                    self.hip.hipGetLastError()
                    break
                self.held.append(p)
        print(f"  filled: {self.free() / GIB:.2f} GiB left", flush=True)
        return self

    def __exit__(self, *exc):
        for p in self.held:
            self.hip.hipFree(p)


def _deck(n, ny, solver, rel, iters, precision="fp64", dt="1e-5"):
    text = decks.reference_deck(n, 1, solver=solver, max_iters=iters).replace(f"y_cells={n}", f"y_cells={ny}")
    extra = "stop_rule=relative\nrel_tol=1e-10\n" if rel else ""
    return text.replace("*endtea", extra + f"precision={precision}\n*endtea").replace("initial_timestep=0.004",
                                                                                       f"initial_timestep={dt}")


@pytest.mark.parametrize("solver,rel,iters", [("cg", False, 9), ("cg", True, 9), ("cg", True, 200),
                                              ("jacobi", False, 107)])
def test_fp64_solvers_need_no_further_field(solver, rel, iters):
    n, ny = 12801, 12800  # 1.22 GiB a field
    print(f"case: {solver}, relative rule {rel}, {iters} iterations, card full", flush=True)
    out = []
    for full in (False, True):
        s = T.Settings.from_text(_deck(n, ny, solver, rel, iters))
        c = T.initialiseapp(s)
        if full:
            with Filler(int(1.05 * GIB)):
                st = T.step(c, s)
                summ = T.fieldsummary(c)
        else:
            st = T.step(c, s)
            summ = T.fieldsummary(c)
        w = c.field("w") if iters == 9 and not rel else None  # scratch for a solve that lacks room
        c.close()
        out.append((summ, (st["iterations"], st["converged"], st["rel_resid"], st["error"]), w))
    assert np.array_equal(out[0][0], out[1][0]), out
    assert out[0][1] == out[1][1], out
    assert np.array_equal(out[0][2], out[1][2])


def test_ragged_fp32_needs_no_further_field():
    n, ny = 17801, 17800  # 1.18 GiB an FP32 field
    print("case: automatic FP32 form on a ragged grid, card full", flush=True)
    out = []
    for full in (False, True):
        s = T.Settings.from_text(_deck(n, ny, "cg", True, 400, "fp32_ir", "1e-7")).set(
            fp32_kernels=_lib.TL_FP32_KERNELS_TWO)
        c = T.initialiseapp(s)
        T.step(c, s)  # the two-kernel form's own arrays
        s.set(fp32_kernels=_lib.TL_FP32_KERNELS_AUTO)
        if full:
            with Filler(int(1.05 * GIB)):
                st = T.step(c, s)
                summ = T.fieldsummary(c)
        else:
            st = T.step(c, s)
            summ = T.fieldsummary(c)
        c.close()
        assert st["converged"] == 1 and st["rel_resid"] <= 1e-10, st
        out.append(summ)
    assert np.max(np.abs(out[0] - out[1]) / np.abs(out[0])) < 1e-9, out
