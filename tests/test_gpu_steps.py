"""The step-record and the generated factorisation and sweeps of the batched kernel on linear networks, against a dense solve.

A network of conductances with one grounded source has a condition number under 1e6 here and converges in one
Newton step, so FP64 agrees to 1e6 times the unit round-off, 1e-10, and mixed precision to the residual test's
1e-12 A over conductances of at least 1e-4 S, 1e-8 V.  Needs the GPU.
"""
import numpy as np
import pytest

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
