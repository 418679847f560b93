"""GPU: field copies through the pinned staging slots.  Every byte of a field
must come back as it was set -- halos, NaN payloads and signed zeros included
-- for one row per field slot, several rows per slot with a remainder, several
slots, and more chunks than slots; and a copy of one field leaves its
neighbours in the allocation order alone."""
import numpy as np
import pytest

import tealeaf_hip as T
from tealeaf_hip import decks

pytestmark = pytest.mark.gpu


# 4 MiB slots: the 540000-column grid is one row per slot, 1001x1201 three
# slots with a remainder, 2000x2650 eleven chunks through eight slots
@pytest.mark.parametrize("nx,ny,hd", [(2, 2, 2), (131, 77, 3), (1001, 1201, 2), (2000, 2650, 2), (540000, 11, 2)])
def test_field_round_trip_bit_exact(nx, ny, hd):
    print(f"case: set_field / field round trip {nx}x{ny} halo {hd}", flush=True)
    text = decks.reference_deck(nx, 1).replace(f"y_cells={nx}", f"y_cells={ny}").replace("halo_depth=2",
                                                                                       f"halo_depth={hd}")
    c = T.initialiseapp(T.Settings.from_text(text))
    before = c.field("u0"), c.field("r")
    rng = np.random.default_rng(nx + ny)
    bits = rng.integers(0, 1 << 64, size=(c.Y, c.X), dtype=np.uint64)  # any pattern, NaNs among them
    bits[0, 0], bits[-1, -1] = 0x7FF0000000000001, 0x8000000000000000
    c.set_field("p", bits.view(np.float64))
    assert np.array_equal(c.field("p").view(np.uint64), bits)
    assert np.array_equal(c.field("u0"), before[0]) and np.array_equal(c.field("r"), before[1])
    c.close()
