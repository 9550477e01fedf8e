"""Ragged f32 products of operands computed while they are staged: light,
one-sided, exponentials and long expressions over the shapes where the
workgroups' rule changes (single k tiles in parts, several, the 16x16 tiling),
against the product of the operands in float64; values past the sides are
computed from the nearest element and dropped, whatever it is."""

import numpy as np
import pytest

from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.ir import F32, Graph


def graph(m, k, n, kind):
    a, b = D.param("a", F32, (m, k)), D.param("b", F32, (k, n))
    if kind != "b":
        a = D.map(D.exp if kind == "exp" else D.neg, a)
    if kind != "a":
        b = D.map(D.exp if kind == "exp" else lambda v: D.add(v, v), b)
    if kind == "long":
        for i in range(30):
            a = D.map(lambda v, i=i: D.add(D.mul(v, D.const(F32, 0.5)), D.const(F32, i / 64)), a)
    return Graph.create("mm", [("c", D.matmul(a, b))])


def grid(g):
    return [(line.split()[2].split("_a")[0], int(line.split()[4])) for line in H.plan(g).splitlines() if line.startswith("kernel")]


@pytest.mark.parametrize("m,k,n,kind,want", [
    (200, 383, 200, "both", ("matmul_mfma_f32", 16 * 6)), (200, 383, 200, "exp", ("matmul_mfma_f32", 16 * 6)),
    (860, 202, 178, "a", ("matmul_mfma_f32", 42 * 4)), (106, 189, 1309, "b", ("matmul_mfma_f32", 42)),
    (106, 189, 1309, "both", ("matmul_mfma_f32", 42 * 3)), (306, 705, 1917, "exp", ("matmul_mfma_f32", 150 * 3)),
    (306, 705, 1917, "both", ("matmul_mfma_f32", 150)), (181, 75, 845, "exp", ("matmul_tiled", 53)),
    (312, 183, 183, "long", ("matmul_tiled", 12)), (1190, 231, 1427, "exp", ("matmul_mfma_f32", 437))])
def test_workgroups(m, k, n, kind, want):
    assert grid(graph(m, k, n, kind))[0] == want


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["a", "b", "both", "exp", "long"])
@pytest.mark.parametrize("m,k,n", [(65, 129, 67), (200, 383, 200), (129, 250, 190), (70, 700, 65), (860, 202, 178), (500, 90, 1300)])
def test_products(device, m, k, n, kind):
    r = np.random.default_rng(m + k + n)
    a, b = r.standard_normal((m, k)).astype(np.float32), r.standard_normal((k, n)).astype(np.float32)
    a[m - 1, ::9], b[::9, n - 1] = -120, -120  # the edge elements are what lanes past the sides compute
    c = H.compile(graph(m, k, n, kind))
    try:
        got = dict(H.run(c, [("a", a), ("b", b)]))["c"].astype(np.float64)
    finally:
        c.release()
    x, y = a.astype(np.float64), b.astype(np.float64)
    x = np.exp(x) if kind == "exp" else -x if kind != "b" else x
    y = np.exp(y) if kind == "exp" else y + y if kind != "a" else y
    if kind == "long":
        for i in range(30):
            x = x * 0.5 + i / 64
    # a rounding a term and a few of the operands (61 of the long one's)
    bound = (k + 70) * 2.0 ** -24 * ((np.abs(x) + (kind == "long")) @ np.abs(y))
    assert (np.abs(got - x @ y) <= bound).all()
