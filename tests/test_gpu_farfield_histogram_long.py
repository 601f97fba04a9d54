"""LDS-histogram far-field binning where a face is longer than its tables of
time products (1024 entries), on either face axis, against the atomic binning:
the same FP32 contributions added in FP64, so they differ by FP64 rounding
only (at most a few 1e5 additions of 1.1e-16 relative to the largest partial
sum, far below 1e-9 of the largest accumulator)."""
import numpy as np
import pytest

from alpineem_amd import decks
from alpineem_amd.solver import Plan, Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ax", [0, 1, 2])
def test_long_faces_equal_atomic(ax):
    cells = [36, 38, 37]
    cells[ax] = 1075
    c = tuple(n // 2 for n in cells)
    dt = decks.courant_dt(1e-3, 1.0)
    deck = decks.Deck(cells=tuple(cells), cell_size=(1e-3, 1e-3, 1e-3), time_steps=60,
                      f_center=decks.gauss_f_center(6.0, dt), phase_centre=c,
                      far_field=[(23.0, 41.0), (90.0, 0.0), (180.0, 0.0)], ports=[decks.Port("z", 50.0, c, (0, 0, 1))])
    plan = Plan.from_text(deck.text())
    v = plan.view
    assert v.ff_hi[ax] - v.ff_lo[ax] + 1 > 1024
    out = {}
    for mode in ("histogram", "atomic"):
        sim = Simulation(plan, ntff=mode)
        sim.run()
        out[mode] = [sim.ntff_raw(w) for w in range(6)]
        sim.close()
    top = max(np.abs(x).max() for x in out["atomic"])
    assert top > 0
    for w in range(6):
        np.testing.assert_allclose(out["histogram"][w], out["atomic"][w], rtol=0, atol=1e-9 * top, err_msg=f"{w}")
