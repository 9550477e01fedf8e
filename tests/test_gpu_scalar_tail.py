"""One-element maps of a reduction's total computed by the kernel that ends
the reduction: chains of them, maps of the total with parameters and with
other totals, over every kernel that ends one (partials folded by one or two
kernels, the split reduction, few and many elements, light and long element
functions), against the oracle and bit for bit against their own kernels."""

import numpy as np
import pytest

import oracle
from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.ir import F32, F64, I32, Graph

pytestmark = pytest.mark.gpu


def graph(dtype, n, heavy, materialised):
    x, k = D.param("x", dtype, (n,)), D.param("k", dtype, ())
    m = D.map(lambda v: D.mul(v, v), x)
    if heavy:
        for i in range(24):
            m = D.map(lambda v, i=i: D.add(D.mul(v, D.const(dtype, 0.5)), D.const(dtype, i / 64)), m)
    s = D.reduce(D.add, D.const(dtype, 1), m)
    mean = D.map(lambda v: D.div(v, D.const(dtype, n)), s)  # the total, then a chain of two uses
    scaled = D.map2(D.mul, mean, k)
    both = D.map2(D.add, scaled, mean)
    top = D.reduce(D.max, D.const(dtype, -1000), x)
    gap = D.map2(D.sub, top, mean)  # two totals, one of them in a tail: its own kernel
    outs = [("s", s), ("mean", mean), ("scaled", scaled), ("both", both), ("top", top), ("gap", gap),
            ("one", D.reshape((1,), scaled))]
    return Graph.create("tail", outs + ([("m", m)] if materialised else []))


def run(g, ins):
    c = H.compile(g)
    try:
        return dict(H.run(c, ins)), [line.split()[2] for line in H.plan(g).splitlines() if line.startswith("kernel")]
    finally:
        c.release()


@pytest.mark.parametrize("materialised", [False, True])
@pytest.mark.parametrize("dtype,heavy", [(F32, False), (F64, False), (I32, False), (F32, True), (F64, True)])
@pytest.mark.parametrize("n", [5, 2049, 100003, 1 << 18, 3000001])
def test_scalar_tail(device, monkeypatch, dtype, n, heavy, materialised):
    r = np.random.default_rng(n)
    x = r.integers(-3, 4, n).astype(dtype.np)  # whole squares, their sum below 2^24: exact
    ins = [("x", x), ("k", np.array(3, dtype.np))]
    g = graph(dtype, n, heavy, materialised)
    got, roles = run(g, ins)
    monkeypatch.setenv("CCHIP_TUNE", "scalar_tail=0")
    own, more = run(g, ins)
    assert (len(roles) < len(more)) == (n > 2048)
    for k in own:
        np.testing.assert_array_equal(got[k], own[k])
    if not heavy:
        for k, e in dict(oracle.run(g, ins)).items():
            np.testing.assert_array_equal(got[k], e)
    else:
        e = x.astype(np.float64) ** 2
        for i in range(24):
            e = e * 0.5 + i / 64
        u = 2.0 ** -24 if dtype is F32 else 2.0 ** -52
        assert abs(float(got["s"]) - 1 - e.sum()) <= (n + 60) * u * (1 + np.abs(e).sum())
