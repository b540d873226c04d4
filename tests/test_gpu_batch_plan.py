"""The planes per block of an ensemble's sweep, planned for the members left."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_autotune_can_keep_the_plan(lulesh_gpu):
    """One small member: its plan cuts it into blocks of a few planes, which
    no fixed count of 8, 16 or 32 comes near, so the tuned batch has it still,
    and the run is the untuned one's."""
    a = lulesh_gpu.Batch([30], stoptime=1e-3)
    b = lulesh_gpu.Batch([30], stoptime=1e-3)
    planned = a.shape()
    assert planned["nz"] < 8
    assert a.autotune(trial_cycles=20) > 0.0
    assert a.shape()["nz"] < 8
    a.run()
    b.run()
    for f in ("x", "xd", "e", "p", "v"):
        assert np.array_equal(a.get(0, f), b.get(0, f))
    a.close()
    b.close()


def test_shape_given_back_stays_planned(lulesh_gpu):
    """The small members stop first; the large one left alone is cut finer
    than all were together, also after get_shape's values were set."""
    sizes = [16] * 60 + [44]
    b = lulesh_gpu.Batch(sizes, stoptime=2e-3)
    s = b.shape()
    s["cycles_per_graph"] = 8
    b.set_shape(**s)
    assert b.shape() == s
    b.run()
    assert b.shape()["nz"] < s["nz"]
    b.close()
    # other planes than the plan's are the caller's, for good
    b = lulesh_gpu.Batch(sizes, stoptime=2e-3)
    s["nz"] += 1
    b.set_shape(**s)
    b.run()
    assert b.shape() == s
    b.close()
