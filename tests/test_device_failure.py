"""Simulations, batches and runs whose HIP calls fail (out of memory, a refused capture)
leave the others, and themselves, as they were: the same fields in the buffers that the
next step reads, late setup still allowed, the next batch and run in order.  On
the CPU, against tests/hip_stub.cpp in place of the HIP runtime; the device
code does nothing there, so a field changes only if a simulation looks at
another buffer.  Each case runs in a process of its own."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FIELDS = ("Ex", "Ey", "Ez", "Hx", "Hy", "Hz")

PRELUDE = f"""
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
sys.path.insert(0, {ROOT!r})
import numpy as np
from alpineem_amd import decks
from alpineem_amd.solver import Batch, Plan, Simulation

FIELDS = {FIELDS!r}
fail = lambda name, nth: stub.stub_fail(name.encode(), ctypes.c_long(nth))

def single_pass_sims(sizes, ntff="histogram", angles=2, steps=4000):
    sims = [Simulation(Plan.from_text(decks.dipole(n=n, steps=steps, angles=angles, arm=6).text()), ntff=ntff)
            for n in sizes]
    assert all(s.single_pass for s in sims)
    return sims

def mark(sims):
    # every member after an odd number of steps, its fields in its second
    # buffer set, marked there only: set_field's copy to the other one fails
    for q, s in enumerate(sims):
        s.run(1, graph=False)
        for r, f in enumerate(FIELDS):
            fail("hipMemcpyAsync", 2)
            assert fails(lambda: s.set_field(f, np.full(s.plan.shape, 10.0 * q + r + 1.0, np.float32)))

def check(sims, what):
    for q, s in enumerate(sims):
        for r, f in enumerate(FIELDS):
            x = s.field(f)
            assert np.all(x == 10.0 * q + r + 1.0), (what, q, f, x.flat[0])

def fails(call):
    try:
        call()
    except RuntimeError as e:
        assert "planted failure" in str(e), e
        return True
    return False
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stub") / "libhipstub.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", out, os.path.join(ROOT, "tests", "hip_stub.cpp")], check=True)
    return out


def run(stub, body):
    r = subprocess.run([sys.executable, "-c", PRELUDE + body, stub], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]


def test_a_failure_is_reported_once(stub):
    """A simulation that could not be created does not fail another one's run."""
    run(stub, """
a = single_pass_sims((36,))[0]
for n in (1, 5, 40):
    fail("hipMalloc", n)
    assert fails(lambda: single_pass_sims((38,)))
    a.run(1, graph=False)
    assert a.steps_done in (1, 2, 3)
assert a.steps_done == 3
""")


@pytest.mark.parametrize("name", ["hipMalloc", "hipMemcpyAsync"])
def test_failed_batch_creation_leaves_members(stub, name):
    """Each allocation and upload of a batch's creation in turn fails."""
    run(stub, f"""
sims = single_pass_sims((36, 38))
mark(sims)
allocs = stub.stub_allocs()
n = 0
while True:
    fail({name!r}, n + 1)
    made = []
    if not fails(lambda: made.append(Batch(sims))):
        break
    n += 1
    check(sims, ({name!r}, n))
    assert stub.stub_allocs() == allocs
    # not a batch's member: its own step is a single pass, into the other buffer set
    sims[0].run(1)
    assert not np.any(sims[0].field("Ez") == 3.0), n
    sims[0].run(1)
    check(sims, ("after two steps of its own", n))
assert n > 10, n
fail("", 0)
check(sims, "created")
made[0].run(4)
check(sims, "run")
""")


@pytest.mark.parametrize("batch", [False, True])
def test_failed_capture_leaves_the_fields(stub, batch):
    """Each call that makes the graph of a run in turn fails, the waits of the
    second stream among them: nothing has run, and the same run then succeeds."""
    run(stub, f"""
sims = single_pass_sims((84, 36) if {batch} else (84,))
mark(sims)
target = Batch(sims) if {batch} else sims[0]
graphs, done = stub.stub_graphs(), sims[0].steps_done
calls = [("hipStreamCreateWithFlags", 1), ("hipStreamBeginCapture", 1), ("hipStreamWaitEvent", 31),
         ("hipEventRecord", 32), ("hipStreamEndCapture", 1), ("hipGraphInstantiate", 1)]
for name, count in calls:
    for n in range(1, count + 1):
        fail(name, n)
        assert fails(lambda: target.run(64)), (name, n)
        check(sims, (name, n))
        assert sims[0].steps_done == done
    assert stub.stub_graphs() - graphs in (0, 1), name   # an attempt's graph goes with the next one
target.run(64)
check(sims, "run")
assert sims[0].steps_done == done + 64
assert stub.stub_graphs() - graphs == 2
""")


def test_a_design_box_is_the_record_box(stub):
    """The design's kernels write record and gradient of its own edges, so
    another record box is refused: its buffers would have another size."""
    run(stub, """
dk, lo, hi = decks.adjoint_deck(n=44, steps=8, box=(5, 6, 4))
plan = Plan.from_text(dk.text())
sim = Simulation(plan, ntff="off")
sim.record_design(lo, [h - 1 for h in hi])       # another box before there is a design: as before
sim = Simulation(plan, ntff="off")
sim.design_box(lo, hi)
for a, b in ((lo, [h - 1 for h in hi]), ([l - 1 for l in lo], hi)):
    try:
        sim.record_design(a, b)
        assert False, (a, b)
    except RuntimeError as e:
        assert "design box" in str(e), e
sim.record_design(lo, hi)
sim.run()
""")
