"""Device evaluation of the batched kernel: every kind of Mos1 and linear element in one assembly, against the oracle.

Stamps differ by the last bits of exp and sqrt: 1e-12 of the entry and of the largest contribution to its row (a
row's entries sum devices of either sign), for the right-hand side of the row's terms a_ij x_j.  Needs the GPU.
"""
import numpy as np
import pytest

from oracle import oracle_py as O
from spice21_amd import _abi as A
from spice21_amd.batch import Batch, Group
from spice21_amd.netlist import Netlist

pytestmark = pytest.mark.gpu


def circuit(n_dev, rng):
    names = [f"n{k}" for k in range(max(3, n_dev // 2))]
    net = Netlist(signals=names)
    node = lambda: "" if rng.random() < 0.15 else names[rng.integers(len(names))]
    models = [net.mos1_model(mos_type=t, vt0=0.25 * (1 - 2 * t), kp=5e-3, tox=1e-7, gamma=g, is_=1e-14, rd=rd, rs=rs)
              for t in (0, 1) for g in (0.0, 0.4) for rd, rs in ((None, None), (50.0, None), (None, 20.0), (10.0, 10.0))]
    inst = net.mos1_inst(w=1e-5, l=1e-6)
    for k in range(n_dev):
        d, g, s = node(), node(), node()
        net.mos1(f"m{k}", d, g, s, s if k % 2 else node(), models[rng.integers(len(models))], inst)
    for k in range(n_dev // 3 + 1):
        net.r(10.0 ** rng.uniform(-4, -2), node(), node())
        net.c(1e-12, node(), node())
        net.i(10.0 ** rng.uniform(-4, -2), node(), node())
    net.v("vs", 1.0, "n0", "")
    return net


@pytest.mark.parametrize("hub", [1, 2])  # every shared slot a hub; only slots of many contributors
@pytest.mark.parametrize("n_dev", [1, 7, 63, 65])
def test_assembly_of_every_kind_of_element(n_dev, hub):
    rng = np.random.default_rng(n_dev)
    cn = circuit(n_dev, rng).to_c()
    b = Batch(Group(cn)).set_hub(hub)
    for trial in range(3):
        x = rng.uniform(-0.5, 0.5, size=cn.n_vars)  # sources and drains change sides from trial to trial
        r, c, v, rhs = b.assemble(x)
        orr, occ, ov, orhs = O.assemble_op(cn, x)
        assert list(r) == list(orr) and list(c) == list(occ)
        row = np.zeros(cn.n_vars)
        np.maximum.at(row, r, np.abs(ov))
        terms = np.abs(orhs)
        np.add.at(terms, r, np.abs(ov * x[c]))
        assert (np.abs(v - ov) <= 1e-12 * (np.abs(ov) + row[r])).all()
        assert (np.abs(rhs - orhs) <= 1e-12 * terms).all()


def check(b, inst, cn, x):
    r, c, v, rhs = b.assemble(x, inst=inst)
    orr, occ, ov, orhs = O.assemble_op(cn, x)
    assert list(r) == list(orr) and list(c) == list(occ)
    row = np.zeros(cn.n_vars)
    np.maximum.at(row, r, np.abs(ov))
    terms = np.abs(orhs)
    np.add.at(terms, r, np.abs(ov * x[c]))
    assert (np.abs(v - ov) <= 1e-12 * (np.abs(ov) + row[r])).all()
    assert (np.abs(rhs - orhs) <= 1e-12 * terms).all()


@pytest.mark.parametrize("fields", [[], [("model", "is_")], [("model", "vt0"), ("model", "is_")]])
def test_junctions_of_instances_with_their_own_parameters(fields):
    """The junctions' saturation currents over the thermal voltage are stored once, or per instance where one overrides the
    current."""
    rng = np.random.default_rng(3)
    net = circuit(9, rng)
    own = [ci for ci, c in enumerate(net.comps) if c[0] == A.S21_COMP_MOS1][::2]
    value = {"is_": lambda: 10.0 ** rng.uniform(-15, -12, size=3), "vt0": lambda: rng.uniform(0.2, 0.3, size=3)}
    over = [(ci, target, field, value[field]()) for ci in own for target, field in fields]
    b = Batch(Group(net.to_c(), 3, over))
    for inst in range(3):
        cn = net.instance(over, inst).to_c()
        for _ in range(2):
            check(b, inst, cn, rng.uniform(-0.5, 0.5, size=cn.n_vars))
