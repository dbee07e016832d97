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


def test_generated_code_leaves_the_lds_to_the_instances():
    """Sixteen chains of 76 stages (mixed precision) share a workgroup only without tables of the factorisation in its
    LDS.  The FP32 factors precondition, so both kernels end within the residual test's 1e-12 A over 1e-6 S or more."""
    nl, over = W.chain_mc(n_inst=4096, stages=76)
    g = Group(nl.to_c(), 4096, over)
    b = Batch(g, precision=MIXED).op()
    assert b.config() == (2, 8, True)
    ref = Batch(g, precision=MIXED).set_jit(-1).op()
    assert (b.status()[0] == 0).all() and (ref.status()[0] == 0).all()
    assert np.abs(b.x() - ref.x()).max() <= 1e-6
