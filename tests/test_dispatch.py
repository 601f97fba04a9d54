"""Which kernels the GPU tests' decks launch: a test that compares a path with
another shows nothing where a rule sends both the same way.  On the CPU: the GPU
tests' own bodies run against tests/hip_stub.cpp, whose kernels do nothing (so
the bodies' checks for non-zero fields may fail) but are counted."""
import pytest

from tests.test_device_failure import run, stub  # noqa: F401  (stub is a fixture)

COUNT = """
def calls(name):
    key = name if name.startswith("hip") else str(len(name)) + name
    stub.stub_calls.restype = ctypes.c_long
    return stub.stub_calls(key.encode())

def body(f, *args):
    stub.stub_forget()
    try:
        f(*args)
    except AssertionError:
        pass
"""


@pytest.mark.parametrize("what", ["", "drude", "sheets", "drude sheets", "drude plane"])
def test_slab_decks(stub, what):  # noqa: F811
    """The one-launch form, but for a Drude box across a TF/SF plane."""
    run(stub, COUNT + f"""
from tests.test_gpu_slab_step import test_slab_step_equals_separate_launches as f
for ax in range(3):
    body(f, ax, (6, 9), {what!r})
    one = {what!r} != "drude plane"
    for k in ("k_h_slab_fix", "k_e_slab_fix"):
        assert (calls(k) > 0) == one, (ax, k)
    assert (calls("k_slab_media") > 0) == (one and {what!r} != ""), ax
    if one:   # not so in the 150 steps of timed phases
        assert calls("k_plane_sums") == 150 + calls("k_h_slab_fix"), ax
""")


def test_ports_beside_the_slabs(stub):  # noqa: F811
    run(stub, COUNT + """
from tests import test_gpu_ports_step as t
for name in t.PORTS:
    body(t.test_ports_equal_oracle, name, 0)
    # (the body ends at the first comparison, of its single-pass run)
    assert calls("k_step_sp") == calls("k_e_slabs") > 0, name
    assert calls("k_ports_h") == 0 and calls("k_step_end") == 0, name
""")


def test_binning_beside_the_next_step(stub):  # noqa: F811
    """The boxes of 76 and 78 cells bin on a second stream, that of 40 does not."""
    run(stub, COUNT + """
from tests import test_gpu_graph_beside as t
for n, wave, beside in ((76, False, True), (78, True, True), (40, False, False)):
    body(t.test_graph_equals_single_steps, n, wave, (160,))
    assert (calls("hipStreamWaitEvent") > 0) == beside, n
    assert calls("hipGraphLaunch") == 10, n
for ntff in ("ordered", "histogram"):
    body(t.test_batch_graph_equals_solo, ntff)
    if ntff == "histogram":      # (the lists of the ordered binning are empty here)
        assert calls("hipStreamWaitEvent") > 0
""")


def test_batches_by_single_passes(stub):  # noqa: F811
    run(stub, COUNT + """
from tests import test_gpu_batch_pass as t
for mixed in (False, True):
    body(t.test_batch_passes_equal_steps_in_place, [2, 7], mixed)
    assert calls("k_step_sp_batch") == (0 if mixed else 8)
    assert (calls("k_e_slabs_batch") > 0) == (not mixed)
    assert calls("k_e_bulk_batch") > 0           # the odd last step, or all
""")


def test_histograms(stub):  # noqa: F811
    """No window is too large for the histogram, which would bin by atomics."""
    run(stub, COUNT + """
from tests import test_gpu_farfield_histogram as t
for name in t.CASES:
    body(t.test_histogram_equals_atomic, name)
    assert calls("k_ntff_hist") > 0 and calls("k_ntff_hist_batch") > 0 and calls("k_ntff_bins") > 0, name
""")


def test_histograms_of_long_faces(stub):  # noqa: F811
    run(stub, COUNT + """
from tests import test_gpu_farfield_histogram_long as t
for ax in range(3):
    body(t.test_long_faces_equal_atomic, ax)
    assert calls("k_ntff_hist") > 0, ax
""")


def test_wide_indices(stub):  # noqa: F811
    run(stub, COUNT + """
from tests import test_gpu_wide_indices as t
calls_of = lambda name: stub.stub_calls(f"{len(name)}{name}It".encode())   # It: of uint16_t
body(t.test_fields_equal_oracle, (70, 45, 39), (2, 2, 2))
assert calls_of("k_step_sp") > 0 and calls_of("k_e_slabs") > 0
for ax in range(3):
    body(t.test_periodic_slab_equals_separate_launches, ax)
    assert calls_of("k_slab_media") > 0 and (calls_of("k_e_bulk_all") > 0) == (ax > 0), ax
body(t.test_batch_with_both_widths)
assert calls("k_step_sp_batch") == 0 and calls_of("k_e_bulk_batch") > 0
body(t.test_gradient)
assert calls_of("k_adj_e") > 0 and calls_of("k_adj_source_gather") > 0
""")


def test_slab_incidence(stub):  # noqa: F811
    run(stub, COUNT + """
from tests import test_gpu_slab_incidence as t
for ax, inc in ((0, (90.0, 180.0)), (1, (90.0, 270.0)), (2, (180.0, 0.0))):
    body(t.test_incidence_equals_separate_launches, ax, inc, 90.0)
    assert calls("k_h_slab_fix") > 0 and calls("k_plane_sums") == 110 + calls("k_h_slab_fix"), ax
""")


def test_run_ahead(stub):  # noqa: F811
    """The host waits once per 64 steps, for the event of 64 steps before."""
    run(stub, COUNT + """
sim = single_pass_sims((36,))[0]
sim.run(128)
for steps in (640, 64):
    stub.stub_forget()
    sim.run(steps)
    assert calls("hipEventSynchronize") == steps // 64 + 1, steps      # and for the end
""")
