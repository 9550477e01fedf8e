"""Whole-tensor scans of an input read at other indices: which templates they
take, and that no pass gathers twice (the pass of totals leaves the values
for the pass of carries), at whole and ragged tiles, with an index error."""

import numpy as np
import pytest

import oracle
from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.ir import F32, F64, I32, I64, Graph

M = 1 << 20


def graph(dtype, n, table, op=D.add, init=0):
    v = D.gather(D.param("i", I32, (n,)), D.param("x", dtype, (table,)))
    return Graph.create("s", [("p", D.scan(op, D.const(dtype, init), v))])


def templates(g):
    return [line.split()[2] for line in H.plan(g).splitlines() if line.startswith("kernel")]


TWO, CHAIN = ["scan_totals", "scan_carry"], ["scan_init", "scan_lookback"]


@pytest.mark.parametrize("dtype,n,table,want", [
    (F32, 2 * M, 4 * M, TWO), (F64, 2 * M, 4 * M, TWO),
    (F32, 2 * M + 1, 4 * M, CHAIN), (F64, 2 * M + 1, 4097, CHAIN), (F64, 2 * M + 1, 4096, TWO),
    (F32, 12 * M, M, TWO), (F32, 12 * M, M + 1, CHAIN), (I64, 12 * M, 5000, CHAIN)], ids=str)
def test_templates(dtype, n, table, want):
    g = graph(dtype, n, table)
    assert templates(g) == want
    # one kernel is given a table (buffer 1) that no CU's cache holds
    used = [line.split(" args ")[1].split() for line in H.plan(g).splitlines() if line.startswith("kernel")]
    assert sum("1" in a for a in used) == (1 if table > 4096 else 2)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, F64, I32, I64], ids=lambda d: d.name)
@pytest.mark.parametrize("n", [M + 1, M + 4096, M + 8190, 3 * M + 5])
def test_sums_of_gathered_values(device, dtype, n):
    r = np.random.default_rng(n)
    i = r.integers(0, 50001, n).astype(np.int32)
    x = r.integers(-3, 4, 50001).astype(dtype.np)  # every partial sum is exact
    c = H.compile(graph(dtype, n, 50001, D.add, 7))
    try:
        np.testing.assert_array_equal(dict(H.run(c, [("i", i), ("x", x)]))["p"], 7 + np.cumsum(x[i], dtype=dtype.np))
        i[n // 2] = 50001
        with pytest.raises(Exception, match="index"):
            H.run(c, [("i", i), ("x", x)])
    finally:
        c.release()
    g = graph(dtype, n, 50001, D.max, 1)
    i[n // 2] = 0
    c = H.compile(g)
    try:
        ins = [("i", i), ("x", x)]
        np.testing.assert_array_equal(dict(H.run(c, ins))["p"], dict(oracle.run(g, ins))["p"])
    finally:
        c.release()


def test_a_scalar_is_not_a_table():
    """A scan of a scaled tensor reads the scalar at one index: it keeps the
    two passes over the tensor itself, in groups of 2 doubles."""
    x, k = D.param("x", F64, (12 * M,)), D.param("k", F64, ())
    g = Graph.create("s", [("p", D.scan(D.add, D.const(F64, 0), D.map(lambda v: D.mul(v, D.const(F64, 2.0)), x)))])
    h = Graph.create("s", [("p", D.scan(D.add, D.const(F64, 0), D.map2(D.mul, x, D.broadcast((12 * M,), k))))])
    assert templates(g) == templates(h) == TWO
    assert all("v[4][2]" in H.source(t) for t in (g, h))


@pytest.mark.parametrize("n,want,group", [(13_107_200, TWO, "v[4][2]"), (13_107_201, CHAIN, "v[8][4]"), (30 * M, CHAIN, "v[8][4]")])
def test_a_small_table_of_doubles(n, want, group):
    """Read in both passes up to 100 MB of sums, in long chains as any table."""
    g = graph(F64, n, 1000)
    assert templates(g) == want and group in H.source(g)
