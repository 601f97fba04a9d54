"""Periodic slab decks: the one-launch form of the terms and copies after the
bulk updates against the separate launches (which time_phases runs), bit for
bit in fields and plane sums, on every slab axis, for small and ragged cross
sections, with Drude media (also across a TF/SF plane, where the separate
launches stay) and thin sheets."""
import numpy as np
import pytest

from alpineem_amd import decks
from alpineem_amd.solver import Plan, Simulation

pytestmark = pytest.mark.gpu

POLES = [((4e10,) * 3, (2e9,) * 3), ((7e10,) * 3, (5e8,) * 3)]
ANGLES = {0: (90.0, 0.0, 90.0), 1: (90.0, 90.0, 90.0), 2: (0.0, 0.0, 270.0)}


@pytest.mark.parametrize("ax", [0, 1, 2])
@pytest.mark.parametrize("cross,what", [((2, 2), ""), ((7, 4), "drude"), ((5, 70), "sheets"), ((65, 3), "drude sheets"),
                                        ((6, 9), "drude plane"), ((16, 16), "drude sheets")])
def test_slab_step_equals_separate_launches(ax, cross, what):
    p, q = [a for a in range(3) if a != ax]
    n = [0, 0, 0]
    n[ax], n[p], n[q] = 64, cross[0], cross[1]
    bounds = [1, 1, 1, 1, 1, 1]
    bounds[2 * ax] = bounds[2 * ax + 1] = 0

    def layer(mid, at, thick):
        start, size = [1, 1, 1], list(n)
        start[ax], size[ax] = at, thick
        return decks.Block(mid, tuple(start), tuple(size))

    mats = [decks.Material(2, (2.0, 3.0, 2.5), (0.01, 0.02, 0.0))]
    objs, sheets = [layer(2, 30, 6)], []
    if "drude" in what:
        mats.append(decks.Material(5, (1.5, 1.5, 1.5), (0.0, 0.0, 0.0), POLES))
        objs.append(layer(5, 12 if "plane" in what else 22, 6))
    if "sheets" in what:
        mats += [decks.SheetMaterial(30, 120.0), decks.SheetMaterial(31, 0.0)]
        sheets = [decks.Sheet("xyz"[ax], 30, 40, (1, 1), cross),
                  decks.Sheet("xyz"[ax], 31, 44, (1, 1), (max(1, cross[0] // 2), max(1, cross[1] - 1)))]
    dt = decks.courant_dt(1e-3, 1.0)
    deck = decks.Deck(cells=tuple(n), cell_size=(1e-3, 1e-3, 1e-3), time_steps=150,
                      f_center=decks.gauss_f_center(10.0, dt), pulse_type=2, boundaries=tuple(bounds),
                      excitation="plane wave", angles=ANGLES[ax], materials=mats, objects=objs, sheets=sheets)
    plan = Plan.from_text(deck.text())
    a, b = Simulation(plan), Simulation(plan)
    a.run(150)
    b.time_phases(150)
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
