"""LDS-histogram far-field binning against the atomic binning.  Both add the
same FP32 contributions in FP64, so they differ by FP64 rounding only: at most
a few 1e5 additions of 1.1e-16 relative to the largest partial sum, far below
1e-9 of the largest accumulator."""
import numpy as np
import pytest

from alpineem_amd import decks
from alpineem_amd.solver import Batch, Plan, Simulation

pytestmark = pytest.mark.gpu

CASES = {
    # every lane in one bin, one bin per row, and rows along either face axis
    "axes": ((44, 44, 44), [(0.0, 0.0), (180.0, 0.0), (90.0, 0.0), (90.0, 90.0)]),
    "planes": ((41, 57, 49), [(30.0, 0.0), (30.0, 90.0), (75.0, 0.0), (2.0, 45.0)]),
    "oblique": ((36, 70, 47), [(23.0, 41.0), (111.0, 200.0), (160.0, 310.0)]),
}


@pytest.mark.parametrize("name", CASES)
def test_histogram_equals_atomic(name):
    cells, angles = CASES[name]
    c = tuple(n // 2 for n in cells)
    dt = decks.courant_dt(1e-3, 1.0)
    deck = decks.Deck(cells=cells, cell_size=(1e-3, 1e-3, 1e-3), time_steps=110, f_center=decks.gauss_f_center(12.0, dt),
                      phase_centre=(c[0] + 2, c[1], c[2] - 3), far_field=angles,
                      ports=[decks.Port("z", 50.0, c, (0, 0, 1))])
    plan = Plan.from_text(deck.text())
    out = {}
    for mode in ("histogram", "atomic", "batch"):
        sim = Simulation(plan, ntff="histogram" if mode == "batch" else mode)
        if mode == "batch":
            other = Simulation(plan, ntff="histogram")
            b = Batch([other, sim])
            b.run()
            b.close()
            other.close()
        else:
            sim.run()
        out[mode] = [sim.ntff_raw(w) for w in range(6)]
        sim.close()
    top = max(np.abs(x).max() for x in out["atomic"])
    assert top > 0
    for mode in ("histogram", "batch"):
        for w in range(6):
            np.testing.assert_allclose(out[mode][w], out["atomic"][w], rtol=0, atol=1e-9 * top, err_msg=f"{mode} {w}")
