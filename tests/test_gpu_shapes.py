"""Launch shapes chosen for a batch: whatever the wavefronts per workgroup, every instance's result is the same.
Needs the GPU."""
import numpy as np
import pytest

from spice21_amd import workloads as W
from spice21_amd.batch import FP64, MIXED, Batch, Group

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("jit", [-1, 1])
@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("n_inst", [1, 225, 257, 1281, 1500, 2049])  # around the CUs, and last rounds of any fill
def test_chosen_shape_gives_the_results_of_one_wavefront_per_workgroup(n_inst, precision, jit):
    nl, over = W.chain_mc(n_inst=n_inst)
    g = Group(nl.to_c(), n_inst, over)
    b = Batch(g, precision=precision).set_jit(jit).op()
    one = Batch(g, precision=precision).set_jit(jit).set_waves(1).op()
    assert np.array_equal(b.status()[0], one.status()[0]) and np.array_equal(b.status()[1], one.status()[1])
    assert np.array_equal(b.x(), one.x())
    if n_inst == 1500:
        assert b.config()[1] * b.config()[0] > 1  # instances share a workgroup
