"""Panel factorisation of the single large instance's dense fronts, against a dense solve.

A complete network of n nodes is one front of n pivots: n covers whole panels of 64 columns, panels that end inside
a 16-column sub-block, and a last panel of one column, above and below the size that one workgroup's LDS holds.
The sweeps take 256 pivots and 256 rows a workgroup: larger networks put several workgroups on one panel, two of them
several fronts in one launch, and random ones children below such a front.
Every node has a conductance of 1e-3 S or more to ground, so the residual test's 1e-12 A bounds a node's error by
1e-9 V.  Needs the GPU.
"""
import numpy as np
import pytest

from spice21_amd import _abi as A
from spice21_amd.batch import FP64, MIXED
from spice21_amd.large import Large
from spice21_amd.netlist import Netlist

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("n", [2, 15, 33, 64, 65, 128, 129, 145, 181, 182, 192, 193, 207, 257, 300])
def test_complete_network_matches_a_dense_solve(n, precision):
    rng = np.random.default_rng(n)
    g = np.tril(10.0 ** rng.uniform(-5, -3, size=(n, n)), -1)
    load, cur = 10.0 ** rng.uniform(-3, -2, size=n), rng.normal(size=n) * 1e-3
    net = Netlist(signals=[f"n{k}" for k in range(n)])
    for a in range(n):
        net.r(load[a], f"n{a}", "")
        net.i(cur[a], f"n{a}", "")
        for b in range(a):
            net.r(g[a, b], f"n{a}", f"n{b}")
    h = Large(net.to_c(), precision=precision).op()
    assert h.status()[0] == 0
    y = -(g + g.T)
    y[np.arange(n), np.arange(n)] = load - y.sum(axis=1)
    v = np.linalg.solve(y, cur)
    off = np.abs(h.x()[:n] - v).max()
    assert off <= 1e-9


def check(n, edges, precision, rng, scale=1.0):
    """A network of the given (a, b) pairs, its conductances, currents and the residual test's current all times
    `scale`, against a dense solve; returns the handle."""
    a, b = (np.array([e[k] for e in edges]) for k in (0, 1))
    g = 10.0 ** rng.uniform(-5, -3, size=len(edges)) * scale
    load, cur = 10.0 ** rng.uniform(-3, -2, size=n) * scale, rng.normal(size=n) * 1e-3 * scale
    net = Netlist(signals=[f"n{k}" for k in range(n)])
    for k in range(n):
        net.r(load[k], f"n{k}", "")
        net.i(cur[k], f"n{k}", "")
    for p, q, c in zip(a, b, g):
        net.r(c, f"n{p}", f"n{q}")
    h = Large(net.to_c(), opts=A.s21_options.default(iabstol=1e-12 * scale), precision=precision).op()
    assert h.status()[0] == 0
    y = np.diag(load)
    np.add.at(y, (a, a), g)
    np.add.at(y, (b, b), g)
    np.subtract.at(y, (a, b), g)
    np.subtract.at(y, (b, a), g)
    assert np.abs(h.x()[:n] - np.linalg.solve(y, cur)).max() <= 1e-9
    return h


@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("n, fronts", [(512, 1), (513, 1), (800, 1), (530, 2)])
def test_sweep_panels_of_several_workgroups(n, fronts, precision):
    rng = np.random.default_rng(n)
    edges = [(f * n + a, f * n + b) for f in range(fronts) for a in range(n) for b in range(a)]
    h = check(fronts * n, edges, precision, rng)
    assert h.structure()["max_front"] == n


@pytest.mark.parametrize("precision", [FP64, MIXED])
def test_large_fronts_with_children(precision):
    rng = np.random.default_rng(1)
    n = 1500
    edges = [(int(rng.integers(k)), k) for k in range(1, n)]
    edges += [tuple(int(v) for v in rng.choice(n, 2, replace=False)) for _ in range(4 * n)]
    s = check(n, edges, precision, rng).structure()
    print(s)
    assert s["max_front"] > 512 and s["levels"] > 1


@pytest.mark.parametrize("scale", [1e-19, 1e21])
@pytest.mark.parametrize("precision", [FP64, MIXED])
@pytest.mark.parametrize("n", [65, 300])
def test_pivots_whose_products_leave_the_range_of_fp32(n, precision, scale):
    check(n, [(a, b) for a in range(n) for b in range(a)], precision, np.random.default_rng(n), scale)


def solve_without_pivoting(y, b, dtype):
    """Elimination of y in panels of 64 without pivoting, each panel's products summed before they are subtracted."""
    a, n = y.astype(dtype), len(y)
    for c in range(0, n, 64):
        e = min(c + 64, n)
        for j in range(c, e):
            a[j + 1:, j] /= a[j, j]
            a[j + 1:, j + 1:e] -= np.outer(a[j + 1:, j], a[j, j + 1:e])
            a[j + 1:e, e:] -= np.outer(a[j + 1:e, j], a[j, e:])
        a[e:, e:] -= a[e:, c:e] @ a[c:e, e:]
    x = b.astype(dtype)
    for j in range(n):
        x[j + 1:] -= a[j + 1:, j] * x[j]
    for j in range(n - 1, -1, -1):
        x[j] /= a[j, j]
        x[:j] -= a[:j, j] * x[j]
    return x.astype(np.float64)


def one_step(g, diag, cur, precision):
    """x after one Newton step from zero (the second iteration's tests are loose) of the complete network with
    conductances g between nodes and the matrix's diagonal diag."""
    n = len(diag)
    net = Netlist(signals=[f"n{k}" for k in range(n)])
    for k in range(n):
        net.r(diag[k] - g[k].sum(), f"n{k}", "")
        net.i(cur[k], f"n{k}", "")
        for q in range(k):
            net.r(g[k, q], f"n{k}", f"n{q}")
    opts = A.s21_options.default(iabstol=1e-9 if precision == FP64 else 2e-7, reltol=10.0)
    h = Large(net.to_c(), opts=opts, precision=precision).op()
    assert h.status()[0] == 0
    return h.x()[:n]


def geo(v):
    return np.exp(np.log(v).mean())


@pytest.mark.parametrize("precision, dtype", [(FP64, np.float64), (MIXED, np.float32)])
def test_error_of_a_nearly_singular_network(precision, dtype):
    """Conductances of 1e-9 to 1e-3 S, grounded through at most 1e-5 S: what the diagonal loses to each subtraction
    decides the error.  It is that of the same elimination in numpy; three times that, since the geometric means of 16
    errors that spread over a factor of ten differ by up to e in three standard deviations."""
    n, off, ref = 300, [], []
    for seed in range(16):
        rng = np.random.default_rng(seed)
        g = np.tril(10.0 ** rng.uniform(-9, -3, size=(n, n)), -1)
        g += g.T
        load, cur = 10.0 ** rng.uniform(-9, -5, size=n), rng.normal(size=n) * 1e-6
        y = np.diag(load + g.sum(axis=1)) - g
        x = np.linalg.solve(y, cur)
        for _ in range(4):
            x = x + np.linalg.solve(y, (cur - y.astype(np.longdouble) @ x).astype(np.float64))
        scale = np.linalg.norm(x)
        off.append(np.linalg.norm(one_step(g, np.diag(y), cur, precision) - x) / scale)
        ref.append(np.linalg.norm(solve_without_pivoting(y, cur, dtype) - x) / scale)
    print(geo(off), geo(ref))
    assert geo(off) <= 3 * geo(ref)


@pytest.mark.parametrize("precision, dtype", [(FP64, np.float64), (MIXED, np.float32)])
@pytest.mark.parametrize("n, diag", [(200, 8.0), (300, 20.0)])
def test_residual_of_networks_with_negative_conductances(n, diag, precision, dtype):
    """Symmetric matrices of normal entries (times 1e-3) with a diagonal that does not dominate: the pivots' blocks are
    ill-conditioned, yet each solve's residual, relative to |y| |x| + |b|, is that of the same elimination in numpy (three
    times it, as above), and every operating point converges."""
    off, ref = [], []
    for seed in range(10):
        rng = np.random.default_rng(seed)
        g = np.zeros((n, n))
        g[np.tril_indices(n, -1)] = rng.normal(size=n * (n - 1) // 2) * 1e-3
        g += g.T
        y, cur = np.diag(np.full(n, diag * 1e-3)) - g, rng.normal(size=n) * 1e-6

        def residual(x):
            r = np.abs(cur - y.astype(np.longdouble) @ x) / (np.abs(y) @ np.abs(x) + np.abs(cur))
            return float(r.max())

        off.append(residual(one_step(g, np.diag(y), cur, precision)))
        ref.append(residual(solve_without_pivoting(y, cur, dtype)))
    print(geo(off), geo(ref))
    assert geo(off) <= 3 * geo(ref)
