"""Analyses repeated on one handle: a kept structure, other initial conditions, and waveforms read in any order give
what a new handle gives, bit for bit.  Needs the GPU."""
import numpy as np
import pytest

from spice21_amd import _abi as A
from spice21_amd import workloads as W
from spice21_amd.batch import FP64, MIXED, Batch, Group
from spice21_amd.large import Large
from spice21_amd.netlist import Netlist

pytestmark = pytest.mark.gpu
TSTEP, TSTOP = 1e-12, 4e-11


def groups():
    out = []
    for k, n_inst in ((5, 3), (9, 70)):  # a few KB of waveform each
        nl = W.ring5(stages=k)
        caps = [(ci, "value", 0, 1e-14 * (1 + np.arange(n_inst) / n_inst)) for ci, c in enumerate(nl.comps) if c[0] == A.S21_COMP_C]
        out.append(Group(nl.to_c(), n_inst, caps))
    return out


def waves(b):
    return [b.wave(g, i) for g in range(len(b.groups)) for i in range(b.groups[g].n_inst)]


@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_repeated_transients_of_a_batch(precision):
    b = Batch(groups(), precision=precision)
    steps = [[("1", 0.5)], [("1", 0.5)], [("1", 0.25)], [("2", 0.25)], None, [("1", 0.25), ("2", 0.5)], [("1", 0.5)]]
    for ics in steps:
        fresh = Batch(groups(), precision=precision)
        if ics is None:
            assert np.array_equal(b.op().x(1), fresh.op().x(1))
            continue
        b.tran(TSTEP, TSTOP, ics)
        fresh.tran(TSTEP, TSTOP, ics)
        assert np.array_equal(b.status(1)[1], fresh.status(1)[1])
        want = [fresh.wave(g, i) for g, i in ((1, 69), (0, 2), (1, 0), (0, 0))]
        got = waves(b)
        for w, k in zip(want, (3 + 69, 2, 3, 0)):
            assert np.array_equal(w, got[k])
    b.tran(TSTEP, TSTOP / 2, steps[0])  # shorter: other buffer, nothing staged before is read
    assert np.array_equal(waves(b)[5], waves(Batch(groups(), precision=precision).tran(TSTEP, TSTOP / 2, steps[0]))[5])


def test_repeated_transients_of_a_single_instance():
    cn = W.power_grid(12, 20, 10, pad_every=6, seed=3).to_c()
    one = Large(cn)
    for ics in ([("g6_6", 0.5)], [("g6_6", 0.5)], [("g6_6", 0.4)], None, [("g6_6", 0.4)]):
        fresh = Large(cn)
        for h in (one, fresh):
            h.op() if ics is None else h.tran(TSTEP, 5.5 * TSTEP, ics=ics)
        assert np.array_equal(one.x(), fresh.x())
        if ics is not None:
            assert np.array_equal(one.wave(), fresh.wave())


def stepped_pair():
    """Two instances of a node that its 1e-3 S or 1e-12 S link pulls to a capacitor's voltage once its initial
    condition ends."""
    net = Netlist(signals=["a", "b"])
    link = net.r(1e-3, "a", "b")
    net.c(1e-6, "b")
    return Group(net.to_c(), 2, [(link, "value", 0, np.array([1e-3, 1e-12]))])


@pytest.mark.parametrize("jit", [-1, 1])
@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_points_that_a_failed_instance_did_not_reach_are_nan(precision, jit):
    """An iteration changes a voltage by at most 1 V and a solve takes at most 100: from 90 V to -90 V the first step
    fails, 300 V are out of the operating point's reach.  The buffer holds the waveforms of the analysis before."""
    b = Batch(stepped_pair(), precision=precision).set_jit(jit)
    for far, near, reached in ((0.9, -0.9, (12, 12)), (90.0, -90.0, (1, 12)), (300.0, -0.9, (0, 0)), (0.9, -0.9, (12, 12))):
        ics = [("a", far), ("b", near)]
        b.tran(1e-9, 11.5e-9, ics)
        want = Batch(stepped_pair(), precision=precision).set_jit(jit).tran(1e-9, 11.5e-9, ics)
        for i, points in enumerate(reached):
            w = b.wave(0, i)
            assert len(w) == 12 and (b.status(0)[0][i] == 0) == (points == 12)
            assert np.isfinite(w[:points]).all() and np.isnan(w[points:]).all()
            assert np.array_equal(w[:points], want.wave(0, i)[:points])


def test_sweep_of_an_instance_without_operating_point_is_nan():
    net = Netlist(signals=["in", "out"])
    v = net.v("vin", 1.0, "in", acm=1.0)
    net.r(1e-3, "in", "out")
    net.c(1e-12, "out")
    b = Batch(Group(net.to_c(), 2, [(v, "value", 0, np.array([1.0, 300.0]))])).ac(1000, 10_000_000, 40)
    assert b.status(0)[0][0] == 0 and b.status(0)[0][1] != 0
    assert np.isfinite(b.wave(0, 0)).all() and np.isnan(b.wave(0, 1)).all()
