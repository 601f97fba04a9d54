"""Decks with more than 256 coefficient tuples, whose cells hold 16-bit
indices: the bulk, single-pass, slab, batch and adjoint kernels of that width.
A cube of small blocks of random anisotropic permittivity gives the tuples."""
import numpy as np
import pytest

from alpineem_amd import decks
from alpineem_amd.solver import Batch, Plan, Simulation
from tests.oracle_ffi import Oracle
from tests.test_gpu_parity import single_pass_deck

pytestmark = pytest.mark.gpu

FIELDS = ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz")


def speckle(deck, start, shape, levels, seed=1):
    """Adds blocks of one cell, each of one of the `levels` per axis."""
    rng = np.random.default_rng(seed)
    for q, at in enumerate(np.ndindex(*shape)):
        deck.materials.append(decks.Material(100 + q, tuple(float(v) for v in rng.choice(levels, 3))))
        deck.objects.append(decks.Block(100 + q, tuple(int(s + a) for s, a in zip(start, at)), (1, 1, 1)))
    return deck


def wide(deck):
    plan = Plan.from_text(deck.text())
    assert plan.view.n_tuple > 256 and plan.view.idx_bytes == 2
    return plan


LEVELS = np.linspace(1.0, 6.0, 11)


@pytest.mark.parametrize("cells", [(70, 45, 39), (36, 66, 52)])
@pytest.mark.parametrize("start", [(2, 2, 2), (24, 16, 14)])     # across the CPML, in the core
def test_fields_equal_oracle(cells, start):
    """Single pass, and core and slabs in one launch, bit for bit."""
    plan = wide(speckle(single_pass_deck(cells, steps=90), start, (6, 6, 6), LEVELS))
    orc = Oracle(plan)
    orc.step(90)
    for sp in (True, False):
        sim = Simulation(plan, single_pass=sp)
        assert sim.single_pass == sp
        sim.run()
        np.testing.assert_array_equal(sim.series("port_v"), orc.series("port_v"), err_msg=f"{sp}")
        for f in FIELDS:
            np.testing.assert_array_equal(sim.field(f), orc.field(f), err_msg=f"{f} {sp}")
        sim.close()


@pytest.mark.parametrize("ax", [0, 1, 2])
def test_periodic_slab_equals_separate_launches(ax):
    """Drude cells and sheets among them, bit for bit; the separate launches
    (timed phases) are within the plane-wave decks' bound of the oracle."""
    p, q = [a for a in range(3) if a != ax]
    n = [9, 9, 9]
    n[ax] = 64
    bounds = [1] * 6
    bounds[2 * ax] = bounds[2 * ax + 1] = 0
    drude = decks.Material(5, (1.5, 1.5, 1.5), (0.0, 0.0, 0.0), [((4e10,) * 3, (2e9,) * 3)])
    start, size = [1, 1, 1], list(n)
    start[ax], size[ax] = 22, 4
    dt = decks.courant_dt(1e-3, 1.0)
    deck = decks.Deck(cells=tuple(n), cell_size=(1e-3, 1e-3, 1e-3), time_steps=120,
                      f_center=decks.gauss_f_center(10.0, dt), pulse_type=2, boundaries=tuple(bounds),
                      excitation="plane wave", angles={0: (90.0, 0.0, 90.0), 1: (90.0, 90.0, 90.0), 2: (0.0, 0.0, 270.0)}[ax],
                      materials=[drude, decks.SheetMaterial(30, 120.0)], objects=[decks.Block(5, tuple(start), tuple(size))],
                      sheets=[decks.Sheet("xyz"[ax], 30, 44, (1, 1), (9, 9))])
    at, shape = [2, 2, 2], [6, 6, 6]
    at[ax] = 30
    plan = wide(speckle(deck, at, shape, LEVELS))
    a, b, orc = Simulation(plan), Simulation(plan), Oracle(plan)
    a.run()
    b.time_phases(120)
    orc.step(120)
    for f in FIELDS:
        x, y = a.field(f), orc.field(f).astype(np.float64)
        np.testing.assert_array_equal(x, b.field(f), err_msg=f)
        assert np.linalg.norm(x - y) <= 5e-5 * np.linalg.norm(y) + 1e-30, f
    a.close()
    b.close()


def test_batch_with_both_widths():
    """Steps in place, each member as alone."""
    cells = [(70, 45, 39), (40, 38, 36)]
    decks_ = [speckle(single_pass_deck(cells[0], steps=65), (24, 16, 14), (6, 6, 6), LEVELS), single_pass_deck(cells[1], steps=65)]
    plans = [Plan.from_text(d.text()) for d in decks_]
    assert [p.view.idx_bytes for p in plans] == [2, 1]
    sims = [Simulation(p) for p in plans]
    batch = Batch(sims)
    batch.run()
    batch.close()
    for p, s in zip(plans, sims):
        ref = Simulation(p)
        ref.run()
        for f in FIELDS:
            np.testing.assert_array_equal(s.field(f), ref.field(f), err_msg=f)
        s.close()
        ref.close()


def test_gradient():
    """Permittivities that differ from 1 by a few roundings (at most 1.5e-6) give
    16-bit indices to a deck that is otherwise the same: fields and gradient move
    by that times the number of periods (at most ten), rounding aside; a wrong
    coefficient moves them by their own size."""
    dk, lo, hi = decks.adjoint_deck(n=44, steps=160, box=(5, 6, 4))
    plans = [Plan.from_text(dk.text())]
    near_one = [float(np.float32(1.0 + q * 2.0 ** -23)) for q in range(13)]
    dk, _, _ = decks.adjoint_deck(n=44, steps=160, box=(5, 6, 4))
    plans.append(wide(speckle(dk, (28, 16, 16), (6, 7, 7), near_one)))
    assert plans[0].view.idx_bytes == 1
    eps = decks.design_permittivity((4, 6, 5))
    out = []
    for p in plans:
        sim = Simulation(p, ntff="off")
        sim.set_objective(30.0, 0.0, 10e9)
        sim.design_box(lo, hi)
        sim.set_design_eps(eps)
        sim.run()
        out.append((sim.objective(), sim.design_gradient()))
        sim.close()
    (f0, g0), (f1, g1) = out
    assert abs(f0) > 0 and np.abs(g0).max() > 0
    assert abs(f1 - f0) <= 1e-3 * abs(f0)
    assert np.abs(g1 - g0).max() <= 1e-3 * np.abs(g0).max()
