"""rp_batch_autotune on batches whose default launch shape is no wave budget at all: helper waves
for a batch of at most one workgroup per compute unit, groups by occupancy for a large one.  What
it settles on has to be as fast as what the batch started with, by the kernels' own times (each
shape's fastest of several runs; the shapes in question are 1.3 times apart), and the way back
from a set budget leads through it."""
import numpy as np
import pytest

from rptunnel import Batch, Pes, specs

pytestmark = pytest.mark.gpu


def _batch(sp, ns, count):
    pols = [dict(n=n, betan=2000.0 / (n + 1), xi=0.5, a=sp.well1, b=sp.well2, dbdl=sp.well2 - sp.well1,
                 stream=1000 * n + k) for n in ns for k in range(count)]
    b = Batch(Pes(sp), sp.mass, pols, 20.0, 1.0, 1e-3, seed=3)
    b.set_path(*specs.linear_path(sp.well1, sp.well2, npath=2))
    b.init_path()
    return b


def _family_ms(b):
    """Each family's fastest launch of 8 steps, launched one after another: by graph the families
    do not overlap, so each time is the family's own."""
    b.set_graphs(True)
    best = np.full(len(b.families()), np.inf)
    for _ in range(12):
        b.run(8)
        best = np.minimum(best, b.last_kernel_ms()[0])
    b.set_graphs(False)
    return best


@pytest.mark.parametrize("ns,count", [([32], 44), ([32, 64], 22), ([32], 5632)])
def test_tuned_is_as_fast_as_untuned(ns, count):
    b = _batch(specs.evb(), ns, count)
    b.set_launch(steps_per_launch=8)
    before = _family_ms(b)
    b.autotune(trial_steps=16)
    b.set_launch(steps_per_launch=8)
    tuned = _family_ms(b)
    assert np.all(tuned <= 1.12 * before), (before, tuned)
    b.set_launch(waves=4)
    b.autotune(trial_steps=16)
    b.set_launch(steps_per_launch=8)
    again = _family_ms(b)
    assert np.all(again <= 1.12 * before), (before, again)
    b.close()
