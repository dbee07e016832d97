"""The step-record and the generated factorisation and sweeps of the batched kernel on linear networks, against a dense solve.

A network of conductances with one grounded source has a condition number under 1e6 here and converges in one
Newton step, so FP64 agrees to 1e6 times the unit round-off, 1e-10, and mixed precision to the residual test's
1e-12 A over conductances of at least 1e-4 S, 1e-8 V.  Small-signal sweeps are compared with the oracle's.  Needs the GPU.
"""
import numpy as np
import pytest

from oracle import oracle_py as O
from spice21_amd.batch import FP64, MIXED, Batch, Group
from spice21_amd.netlist import Netlist

pytestmark = pytest.mark.gpu


def network(kind, n, rng):
    """Edges (a, b) of a network on nodes 0..n-1, node 0 the source; every node has a path to it."""
    if kind == "line":  # one level per node
        return [(k, k + 1) for k in range(n - 1)]
    if kind == "star":  # one wide level, one long row
        return [(0 if k % 2 else 1, k) for k in range(2, n)] + [(0, 1)]
    if kind == "complete":  # rows of more entries than a record holds
        return [(a, b) for a in range(n) for b in range(a)]
    return [(int(rng.integers(k)), k) for k in range(1, n)] + [tuple(rng.choice(n, 2, replace=False)) for _ in range(n)]


def check(kind, n, ipw, precision, jit=-1):
    rng = np.random.default_rng(n)
    net = Netlist(signals=[f"n{k}" for k in range(n)])
    edges = network(kind, n, rng)
    ninst = 1 if n == 560 else 5  # 560: the records do not fit beside the instance, the level tables run
    g = 10.0 ** rng.uniform(-4, -2, size=(ninst, len(edges) + n))
    over = [(net.r(1.0, f"n{a}", f"n{b}"), "value", 0, g[:, k]) for k, (a, b) in enumerate(edges)]
    over += [(net.r(1.0, f"n{k}", ""), "value", 0, g[:, len(edges) + k]) for k in range(n)]  # a load at every node
    net.v("vs", 1.0, "n0", "")
    b = Batch(Group(net.to_c(), ninst, over), precision=precision)
    if ipw:
        b.set_ipw(ipw)
    b.set_jit(jit)
    x = b.op().x()
    assert (b.status()[0] == 0).all()
    for i in range(ninst):
        y = np.zeros((n, n))
        for k, (p, q) in enumerate(edges):
            y[[p, q], [p, q]] += g[i, k]
            y[[p, q], [q, p]] -= g[i, k]
        y[np.arange(n), np.arange(n)] += g[i, len(edges):]
        v = np.ones(n)
        v[1:] = np.linalg.solve(y[1:, 1:], -y[1:, 0])
        off = np.abs(x[i, :n] - v).max()
        assert off <= (1e-10 if precision == FP64 else 1e-8)


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("ipw", [1, 16])  # 64 lanes per instance, and 4: fewer than the widest step's records
@pytest.mark.parametrize("kind, n", [("line", 2), ("line", 3), ("line", 70), ("line", 560), ("star", 40),
                                     ("complete", 6), ("complete", 11), ("random", 23), ("random", 64)])
def test_linear_networks_match_a_dense_solve(kind, n, ipw, precision):
    check(kind, n, 0 if n == 560 else ipw, precision)


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("kind, n", [("line", 2), ("line", 70), ("star", 40), ("complete", 11), ("random", 23)])
def test_generated_factorisation_of_linear_networks(kind, n, precision):
    """Written-out steps: chunks of long rows, values older than the locals kept, rows without L entries."""
    check(kind, n, 0, precision, jit=1)


def common_source(devices):
    """A stage whose output node's row has 2 * devices + 3 entries and no node of more than four contributors for up
    to three devices: gates and sources of their own, the bulks on a body supply."""
    net = Netlist(signals=["vdd", "out", "bb", "in"])
    net.v("vvdd", 1.2, "vdd")
    net.v("vbb", -0.1, "bb")
    net.v("vin", 0.6, "in", acm=1.0)
    model = net.mos1_model(mos_type=0, vt0=0.3, kp=5e-3, tox=2e-9, gamma=0.3, is_=1e-14)
    inst = net.mos1_inst(w=1e-6, l=1e-6)
    net.r(1e-3, "vdd", "out")
    for k in range(devices):
        net.r(1e-3 * (1 + k), "in", f"g{k}")
        net.r(2e-3 * (1 + k), f"s{k}")
        net.c(1e-12, f"s{k}")
        net.mos1(f"m{k}", "out", f"g{k}", f"s{k}", "bb", model, inst)
    return net


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("jit", [-1, 1])
@pytest.mark.parametrize("devices", [2, 3, 4, 8])  # no hub cells and no split row; no hub cells; hub cells and split rows
def test_small_signal_sweep_with_split_rows(devices, jit, precision):
    cn = common_source(devices).to_c()
    b = Batch(Group(cn, 3), precision=precision).set_jit(jit).ac(1000, 10_000_000_000, 60)
    assert (b.status()[0] == 0).all()
    f, want, _ = O.ac(cn, 1000, 10_000_000_000, 60, max_pts=100)
    assert np.array_equal(b.axis(), f)
    for i in range(3):  # the residual test's 1e-9 A over conductances of 1e-3 S or more leaves mixed precision 1e-6 V
        assert np.abs(b.wave(0, i) - want).max() <= (1e-12 if precision == FP64 else 1e-6)


def mesh(m, n_inst, rng):
    """m x m nodes; returns the group and each instance's expected voltages (all instances alike)."""
    n = m * m
    edges = [(a * m + b, a * m + b + 1) for a in range(m) for b in range(m - 1)]
    edges += [(a * m + b, a * m + b + m) for a in range(m - 1) for b in range(m)]
    net = Netlist(signals=[f"n{k}" for k in range(n)])
    y = np.zeros((n, n))
    for a, b in edges:
        g = 10.0 ** rng.uniform(-4, -2)
        net.r(g, f"n{a}", f"n{b}")
        y[[a, b], [a, b]] += g
        y[[a, b], [b, a]] -= g
    for k in range(n):
        net.r(1e-4, f"n{k}", "")
    y[np.arange(n), np.arange(n)] += 1e-4
    net.v("vs", 1.0, "n0", "")
    v = np.ones(n)
    v[1:] = np.linalg.solve(y[1:, 1:], -y[1:, 0])
    return Group(net.to_c(), n_inst), v


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("meshes", [((10, 1), (12, 1)), ((10, 2), (4, 3), (12, 1)), ((7, 1),), ((10, 1),)])
def test_meshes_whose_step_records_take_much_of_the_lds(meshes, precision):
    """Groups that fit together only when some of them have level tables (10 x 10 beside 12 x 12), and groups alone."""
    rng = np.random.default_rng(5)
    made = [mesh(m, k, rng) for m, k in meshes]
    b = Batch([g for g, _ in made], precision=precision).set_hub(2).set_jit(-1).op()
    for k, (g, v) in enumerate(made):
        assert (b.status(k)[0] == 0).all()
        assert np.abs(b.x(k)[:, :len(v)] - v).max() <= (1e-10 if precision == FP64 else 1e-8)


@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_tables_follow_the_launch(precision):
    """Step records of a 10 x 10 mesh leave room for one FP64 instance in the LDS: a large batch has level tables, which
    leave room for several, and the choice is made again when the launch's settings change."""
    rng = np.random.default_rng(6)
    g, v = mesh(10, 2048, rng)
    b = Batch(g, precision=precision).set_jit(-1)
    for waves, ipw in ((0, 0), (1, 1), (0, 2), (0, 0)):
        b.set_waves(waves).set_ipw(ipw).op()
        assert (b.status(0)[0] == 0).all()
        assert np.abs(b.x(0)[:, :len(v)] - v).max() <= (1e-10 if precision == FP64 else 1e-8)
        assert b.config()[0] * b.config()[1] > 1 or (waves, ipw) == (1, 1)
