"""Ordered far-field binning at the ends of what a deck may ask of the
contributor lists: a phase centre so far outside the grid that the retarded
time is a small difference of large terms, and lists that pass their limit of
memory only by their padding."""
import numpy as np
import pytest

from alpineem_amd import decks
from alpineem_amd.solver import Plan, Simulation
from tests.oracle_ffi import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lists", [True, False])
@pytest.mark.parametrize("off,phis", [(1000, [45.0, 45.5]), (100000, [45.02, 45.1, 45.2, 45.3]), (400000, [45.01, 45.06])])
def test_far_phase_centre_equals_oracle(off, phis, lists):
    """Bit for bit: every face cell contributes to the bins that the
    reference's FP32 time gives it."""
    dt = decks.courant_dt(1e-3, 1.0)
    deck = decks.Deck(cells=(36, 38, 40), cell_size=(1e-3, 1e-3, 1e-3), time_steps=120,
                      f_center=decks.gauss_f_center(12.0, dt), phase_centre=(18 + off, 18 - off, 20),
                      far_field=[(90.0, p) for p in phis], ports=[decks.Port("z", 50.0, (18, 19, 20), (0, 0, 1))])
    plan = Plan.from_text(deck.text())
    orc = Oracle(plan)
    orc.step(plan.time_steps)
    sim = Simulation(plan, ntff_lists=lists)
    sim.run()
    for w in range(6):
        ref = orc.ntff_raw(w)
        assert all(np.any(r != 0) for r in ref)
        np.testing.assert_array_equal(sim.ntff_raw(w), ref, err_msg=f"accumulator {w}")
    sim.close()


def test_lists_past_their_limit_by_padding():
    """A ground-plane deck, whose far field only the lists bin, with 2,600
    directions about 5 degrees off the axis: 0.47 MB a direction without padding,
    2.0 MB with it, against a limit of 4 GiB.  A few of the directions equal
    those of a deck that has only these, whose lists are grouped."""
    def deck(angles):
        dt = decks.courant_dt(1e-3, 1.0)
        return decks.Deck(cells=(60, 60, 60), cell_size=(1e-3, 1e-3, 1e-3), time_steps=60, igp=("-z", 16),
                          f_center=decks.gauss_f_center(8.0, dt), excitation="plane wave", angles=(180.0, 0.0, 90.0),
                          pulse_type=2, phase_centre=(30, 30, 30), far_field=angles)

    n = 2600
    every = [(5.0 + 0.1 * float(np.sin(q)), 0.001 * q) for q in range(n)]
    some = [0, 1, 1300, n - 1]
    out = []
    for angles, pick in ((every, some), ([every[q] for q in some], range(len(some)))):
        sim = Simulation(Plan.from_text(deck(angles).text()))
        sim.run()
        sim.finalize()
        out.append(np.array([[sim.series(k, q) for k in ("e_theta", "e_phi")] for q in pick]))
        sim.close()
    assert all(np.any(x != 0) for x in out[1])
    np.testing.assert_array_equal(out[0], out[1])
