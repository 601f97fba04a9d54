"""Lumped ports in the single-pass step (beside the slabs' E phase) and in the
separate launches, against the oracle bit for bit: every gap axis, gaps of one
cell, of more loop terms than a wave has lanes, and several ports."""
import numpy as np
import pytest

from alpineem_amd import decks
from alpineem_amd.solver import Plan, Simulation
from tests.oracle_ffi import Oracle

pytestmark = pytest.mark.gpu

PORTS = {
    "one_cell": [decks.Port("z", 50.0, (20, 19, 21), (0, 0, 1))],
    "axes": [decks.Port("x", 50.0, (15, 16, 20), (2, 1, 0)), decks.Port("y", 75.0, (20, 15, 18), (0, 3, 2)),
             decks.Port("z", 30.0, (24, 22, 16), (1, 0, 4))],
    "long": [decks.Port("z", 50.0, (15, 16, 17), (2, 2, 12)), decks.Port("x", 50.0, (24, 17, 15), (5, 1, 2))],
    "five": [decks.Port("z", 50.0, (14 + 3 * q, 20, 20), (0, 0, 1 + q % 2)) for q in range(5)],
}


@pytest.mark.parametrize("angles", [0, 1])
@pytest.mark.parametrize("name", PORTS)
def test_ports_equal_oracle(name, angles):
    dt = decks.courant_dt(1e-3, 1.0)
    deck = decks.Deck(cells=(40, 38, 42), cell_size=(1e-3, 1e-3, 1e-3), time_steps=130,
                      f_center=decks.gauss_f_center(12.0, dt), excitation_port=1, phase_centre=(20, 19, 21),
                      far_field=[(50.0, 20.0)] * angles, ports=PORTS[name],
                      materials=[decks.Material(3, (2.5, 2.5, 2.5), (0.02, 0.02, 0.02))],
                      objects=[decks.Block(3, (14, 14, 14), (10, 12, 9))])
    plan = Plan.from_text(deck.text())
    orc = Oracle(plan)
    orc.step(plan.time_steps)
    for sp in (True, False):
        sim = Simulation(plan, single_pass=sp)
        assert sim.single_pass == sp
        sim.run(57)
        sim.run(73)
        for q in range(len(PORTS[name])):
            np.testing.assert_array_equal(sim.series("port_v", q), orc.series("port_v", q), err_msg=f"V {q} {sp}")
        for f in ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz"):
            np.testing.assert_array_equal(sim.field(f), orc.field(f), err_msg=f"{f} {sp}")
        sim.close()
