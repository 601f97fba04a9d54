"""Periodic slab decks in the one-launch form of their terms and copies, for
waves from either side and of every polarisation, against the separate launches
(which time_phases runs), bit for bit in fields and plane sums."""
import numpy as np
import pytest

from alpineem_amd import decks
from alpineem_amd.solver import Plan, Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pol", [0.0, 90.0, 210.0])
@pytest.mark.parametrize("ax,incidence", [(0, (90.0, 0.0)), (0, (90.0, 180.0)), (1, (90.0, 90.0)), (1, (90.0, 270.0)),
                                          (2, (0.0, 0.0)), (2, (180.0, 0.0))])
def test_incidence_equals_separate_launches(ax, incidence, pol):
    n = [7, 9, 6]
    n[ax] = 60
    bounds = [1] * 6
    bounds[2 * ax] = bounds[2 * ax + 1] = 0
    start, size = [1, 1, 1], list(n)
    start[ax], size[ax] = 28, 5
    dt = decks.courant_dt(1e-3, 1.0)
    deck = decks.Deck(cells=tuple(n), cell_size=(1e-3, 1.25e-3, 0.8e-3), time_steps=110,
                      f_center=decks.gauss_f_center(9.0, dt), pulse_type=1, boundaries=tuple(bounds),
                      excitation="plane wave", angles=incidence + (pol,),
                      materials=[decks.Material(2, (2.0, 3.0, 2.5), (0.01, 0.02, 0.0)), decks.SheetMaterial(30, 200.0)],
                      objects=[decks.Block(2, tuple(start), tuple(size))],
                      sheets=[decks.Sheet("xyz"[ax], 30, 37, (1, 1), tuple(v for a, v in enumerate(n) if a != ax))])
    plan = Plan.from_text(deck.text())
    a, b = Simulation(plan), Simulation(plan)
    a.run(110)
    b.time_phases(110)
    for f in ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz"):
        x = a.field(f)
        assert np.isfinite(x).all()
        np.testing.assert_array_equal(x, b.field(f), err_msg=f)
    assert any(np.any(a.field(f) != 0) for f in ("Ex", "Ey", "Ez"))
    a.finalize()
    b.finalize()
    for k in ("reflected", "transmitted"):
        np.testing.assert_array_equal(a.series(k), b.series(k), err_msg=k)
    a.close()
    b.close()
