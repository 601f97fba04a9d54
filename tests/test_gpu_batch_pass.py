"""A batch whose members all admit the single pass steps two at a time between
their buffer sets, a last step in place; other batches step in place.  Either
way a member's fields, port and far-field series are bit-identical to a run of
its own in place."""
import numpy as np
import pytest

from alpineem_amd.solver import Batch, Plan, Simulation
from tests.test_gpu_parity import single_pass_deck

pytestmark = pytest.mark.gpu

CELLS = [(70, 45, 39), (36, 66, 52), (40, 38, 36)]


# one in place; pairs; graphs with an odd rest; an odd run before graphs
@pytest.mark.parametrize("runs", [[1], [2, 7], [63], [3, 64]])
@pytest.mark.parametrize("mixed", [False, True])
def test_batch_passes_equal_steps_in_place(runs, mixed):
    steps = sum(runs)
    texts = [single_pass_deck(c, steps=steps).text() for c in CELLS]
    sims = [Simulation(Plan.from_text(t), planes=p, single_pass=not (mixed and q == 1))
            for q, (t, p) in enumerate(zip(texts, (0, 3, 0)))]
    if not mixed:
        assert all(s.single_pass for s in sims)
    batch = Batch(sims)
    for n in runs:
        batch.run(n)
    batch.close()
    for t, s in zip(texts, sims):
        ref = Simulation(Plan.from_text(t), single_pass=False)
        ref.run(steps)
        for x in (s, ref):
            x.finalize()
        for comp in ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz"):
            np.testing.assert_array_equal(s.field(comp), ref.field(comp), err_msg=comp)
        for q in range(s.plan.view.n_ports):
            for kind in ("port_v", "port_i"):
                np.testing.assert_array_equal(s.series(kind, q), ref.series(kind, q), err_msg=kind)
        for q in range(s.plan.view.n_angles):
            for kind in ("e_theta", "e_phi"):
                np.testing.assert_array_equal(s.series(kind, q), ref.series(kind, q), err_msg=kind)
        s.close()
        ref.close()


def test_members_in_different_buffer_sets():
    """Members enter a batch after an odd and an even number of steps."""
    texts = [single_pass_deck(c, steps=40).text() for c in CELLS[1:]]
    sims = [Simulation(Plan.from_text(t)) for t in texts]
    sims[0].run(5)
    sims[1].run(4)
    Batch(sims).run(35)
    sims[1].run(1)
    for t, s in zip(texts, sims):
        ref = Simulation(Plan.from_text(t), single_pass=False)
        ref.run(40)
        for comp in ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz"):
            np.testing.assert_array_equal(s.field(comp), ref.field(comp), err_msg=comp)
