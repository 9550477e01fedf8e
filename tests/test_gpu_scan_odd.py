"""Scans of rows whose length is no multiple of a thread's group (2 or 4
elements), at the edges of groups, slices and tiles, in every tile template:
one tile a row, the look-back and the two passes of totals and carries.
Integers, max and min bit for bit against the oracle; float sums within
the bound of any summation order, n u sum|x|, of a long double scan."""

import numpy as np
import pytest

import oracle
from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.ir import F32, F64, I32, I64, Graph

pytestmark = pytest.mark.gpu


def templates(g):
    return [line.split()[2] for line in H.plan(g).splitlines() if line.startswith("kernel")]


def run(g, inputs):
    c = H.compile(g)
    try:
        return dict(H.run(c, inputs))
    finally:
        c.release()


def data(dtype, shape, seed):
    r = np.random.default_rng(seed)
    if dtype in (I32, I64):
        return r.integers(-1000, 1000, shape).astype(dtype.np)
    return r.standard_normal(shape).astype(dtype.np)


def check_sum(got, x, init, dtype):
    e = np.cumsum(x.astype(np.longdouble), axis=-1) + init
    u = 2.0 ** -24 if dtype is F32 else 2.0 ** -53
    n = x.shape[-1]
    assert (np.abs(got - e) <= n * u * (np.cumsum(np.abs(x.astype(np.longdouble)), axis=-1) + abs(init))).all()


def graph(dtype, shape, op, init):
    x = D.param("x", dtype, shape)
    ini = D.const(dtype, init)
    f = D.scan if len(shape) == 1 else D.scan_rows
    r = D.reduce if len(shape) == 1 else D.reduce_rows
    low = -(1 << 30) if dtype in (I32, I64) else -1e30
    return Graph.create("s", [("p", f(op, ini, x)), ("end", r(op, ini, x)), ("max", r(D.max, D.const(dtype, low), x))])


def check(dtype, shape, op, init, seed):
    g, x = graph(dtype, shape, op, init), data(dtype, shape, seed)
    got = run(g, [("x", x)])
    if dtype in (F32, F64) and op is D.add:
        check_sum(got["p"], x, init, dtype)
    else:
        exp = dict(oracle.run(g, [("x", x)]))
        np.testing.assert_array_equal(got["p"], exp["p"])
    np.testing.assert_array_equal(got["end"], got["p"][..., -1])
    np.testing.assert_array_equal(got["max"], x.max(axis=-1))


@pytest.mark.parametrize("dtype", [F32, F64, I32, I64], ids=lambda d: d.name)
@pytest.mark.parametrize("shape", [(3, 65), (3, 67), (5, 2047), (5, 2049), (4, 4093), (4, 8191), (3, 16383), (1500, 3001)],
                         ids=str)
def test_one_tile_a_row(device, dtype, shape):
    assert any(t.startswith("scan_tile") for t in templates(graph(dtype, shape, D.add, 0)))
    check(dtype, shape, D.add, 3, shape[1])
    check(dtype, shape, D.max, 1, shape[1] + 1)


@pytest.mark.parametrize("dtype", [F32, F64, I32, I64], ids=lambda d: d.name)
@pytest.mark.parametrize("shape", [(3, 26625), (2, 26627), (2, 40001), (5, 300001), (70, 27001), (50003,), (1 << 20,)], ids=str)
def test_look_back(device, dtype, shape):
    assert "scan_lookback" in templates(graph(dtype, shape, D.add, 0))
    check(dtype, shape, D.add, 2, shape[-1])
    check(dtype, shape, D.min, -5, shape[-1] + 1)


@pytest.mark.parametrize("knobs", ["", "scan_carry=0"])
@pytest.mark.parametrize("dtype", [F32, F64, I32, I64], ids=lambda d: d.name)
@pytest.mark.parametrize("n", [(1 << 20) + 1, (1 << 20) + 4096, (1 << 20) + 8191, 3000001])
def test_totals_and_carries(device, monkeypatch, dtype, n, knobs):
    monkeypatch.setenv("CCHIP_TUNE", knobs)
    t = templates(graph(dtype, (n,), D.add, 0))
    assert ("scan_carry" in t) == (not knobs) and ("scan_lookback" in t) == bool(knobs)
    check(dtype, (n,), D.add, 7, n)
    check(dtype, (n,), D.max, -3, n + 1)


@pytest.mark.parametrize("dtype", [F32, F64])
def test_totals_and_carries_of_an_expression(device, dtype):
    """The input is computed in both passes; NaN and infinities reach the
    elements after them and no others, -0 stays first in a max."""
    n = (1 << 20) + 77
    x, i = data(dtype, (n,), 4), np.random.default_rng(3).integers(0, n, n).astype(np.int32)
    x[n - 100], x[n - 50] = np.inf, np.nan
    v = D.map2(D.mul, D.gather(D.param("i", I32, (n,)), D.param("x", dtype, (n,))), D.param("y", dtype, (n,)))
    g = Graph.create("s", [("p", D.scan(D.max, D.const(dtype, -1e30), v))])
    assert templates(g) == ["scan_totals", "scan_carry"]
    ins = [("i", i), ("x", x), ("y", data(dtype, (n,), 5))]
    np.testing.assert_array_equal(run(g, ins)["p"], dict(oracle.run(g, ins))["p"])


@pytest.mark.parametrize("n", [(1 << 20) + 5])
def test_a_combine_that_needs_its_order_keeps_the_look_back(device, n):
    """f(a, b) = b where b is not zero, else a: associative, not
    commutative; the last non-zero value so far."""
    x = data(I32, (n,), 8) * (np.arange(n) % 37 == 0)
    last = lambda a, b: D.select(D.ne(b, D.const(I32, 0)), b, a)  # noqa: E731
    g = Graph.create("s", [("p", D.scan(last, D.const(I32, 9), D.param("x", I32, (n,))))])
    assert "scan_lookback" in templates(g)
    x = x.astype(np.int32)
    np.testing.assert_array_equal(run(g, [("x", x)])["p"], dict(oracle.run(g, [("x", x)]))["p"])
