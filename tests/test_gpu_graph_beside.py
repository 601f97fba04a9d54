"""Runs in graphs, where the far-field binning of a step runs beside the next
step, against the same steps enqueued one by one on one stream: bit for bit in
fields and ordered accumulators, for run lengths that end inside a graph, on
it and in several calls."""
import numpy as np
import pytest

from alpineem_amd import decks
from alpineem_amd.solver import Batch, Plan, Simulation

pytestmark = pytest.mark.gpu

FIELDS = ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz")


def deck(n, wave):
    c = n // 2
    if wave:
        return decks.pec_sphere(n=n, steps=160, radius=6, angles=[(180.0, 0.0), (37.0, 61.0)])
    return decks.dipole(n=n, steps=160, angles=5, arm=8)


@pytest.mark.parametrize("runs", [(160,), (49, 47, 64), (1, 48, 15, 96)])
@pytest.mark.parametrize("n,wave", [(76, False), (78, True), (40, False)])
def test_graph_equals_single_steps(n, wave, runs):
    plan = Plan.from_text(deck(n, wave).text())
    a, b = Simulation(plan), Simulation(plan)
    for k in runs:
        a.run(k)
        b.run(k, graph=False)
        for w in range(6):
            np.testing.assert_array_equal(a.ntff_raw(w), b.ntff_raw(w), err_msg=f"accumulator {w} after {a.steps_done}")
    for f in FIELDS:
        np.testing.assert_array_equal(a.field(f), b.field(f), err_msg=f)
    a.close()
    b.close()


@pytest.mark.parametrize("ntff", ["ordered", "histogram"])
def test_batch_graph_equals_solo(ntff):
    plans = [Plan.from_text(deck(n, w).text()) for n, w in ((76, False), (41, False), (78, True))]
    solo = [Simulation(p, ntff=ntff) for p in plans]
    members = [Simulation(p, ntff=ntff) for p in plans]
    batch = Batch(members)
    for k in (49, 111):
        batch.run(k)
        for s in solo:
            s.run(k, graph=False)
    batch.close()
    for s, m in zip(solo, members):
        for w in range(6):
            x, y = s.ntff_raw(w), m.ntff_raw(w)
            if ntff == "ordered":
                np.testing.assert_array_equal(x, y)
            else:
                np.testing.assert_allclose(x, y, rtol=0, atol=1e-12 * np.abs(x).max())
        for f in FIELDS:
            np.testing.assert_array_equal(s.field(f), m.field(f), err_msg=f)
        s.close()
        m.close()
