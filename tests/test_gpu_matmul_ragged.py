"""Matrix products on the matrix cores whose sides are no multiple of the
tile: every remainder of a tile edge, both tile sizes, each operand mode
(a buffer, a transposed buffer, a fused expression), against the product in
long double (f64) or float64 (f32) within the bound every summation order
of K fused steps meets, (K + 2) u sum |a||b|."""

import numpy as np
import pytest

from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.ir import F32, F64, Graph

pytestmark = pytest.mark.gpu


def graph(m, k, n, dtype, mode):
    if mode == "t":
        a, b = D.transpose(D.param("a", dtype, (k, m))), D.transpose(D.param("b", dtype, (n, k)))
    else:
        a, b = D.param("a", dtype, (m, k)), D.param("b", dtype, (k, n))
    if mode == "f":
        a, b = D.map(D.neg, a), D.map(lambda v: D.add(v, v), b)
    return Graph.create("mm", [("c", D.matmul(a, b))])


def run(g, a, b):
    c = H.compile(g)
    try:
        return dict(H.run(c, [("a", a), ("b", b)]))["c"]
    finally:
        c.release()


def roles(g):
    return [line.split()[2] for line in H.plan(g).splitlines() if line.startswith("kernel")]


SIZES = [(32, 48, 32), (33, 49, 35), (63, 64, 65), (64, 65, 64), (65, 127, 129), (127, 63, 128), (200, 129, 61),
         (1, 48, 1)]
BIG = [(F32, 1790, 70, 1930), (F64, 1100, 70, 1190)]  # past the line of the large tile


@pytest.mark.parametrize("mode", ["d", "t", "f"])
@pytest.mark.parametrize("dtype,m,k,n", [(d,) + s for d in (F32, F64) for s in SIZES] + BIG)
def test_ragged_product(device, dtype, m, k, n, mode):
    rng = np.random.default_rng(m * 1000003 + k * 1009 + n)
    a, b = rng.standard_normal((m, k)).astype(dtype.np), rng.standard_normal((k, n)).astype(dtype.np)
    g = graph(m, k, n, dtype, mode)
    assert any(r.startswith("matmul_mfma_" + dtype.name) for r in roles(g)) == (min(m, n) >= 32)
    got = run(g, np.ascontiguousarray(a.T) if mode == "t" else a, np.ascontiguousarray(b.T) if mode == "t" else b)
    wide = np.longdouble if dtype is F64 and m < 1000 else np.float64
    aw, bw = a.astype(wide), b.astype(wide)
    if mode == "f":
        aw, bw = -aw, bw + bw
    u = 2.0 ** -24 if dtype is F32 else 2.0 ** -53
    bound = (k + 2) * u * (np.abs(aw) @ np.abs(bw))
    if wide is np.float64 and dtype is F64:
        bound = 2 * bound  # the float64 reference has as many roundings
    assert (np.abs(got - aw @ bw) <= bound).all()


@pytest.mark.parametrize("mode", ["d", "t", "f"])
@pytest.mark.parametrize("dtype", [F32, F64])
def test_ragged_product_keeps_infinities_and_nans_in_their_rows_and_columns(device, dtype, mode):
    """What the loads past an edge pick up (the next row's first values)
    reaches no stored output."""
    m, k, n = 70, 75, 90
    rng = np.random.default_rng(9)
    a, b = rng.uniform(1, 2, (m, k)).astype(dtype.np), rng.uniform(1, 2, (k, n)).astype(dtype.np)
    a[5, 0], a[30, k - 1], b[0, 7], b[k - 1, 41] = np.inf, np.nan, -np.inf, np.inf
    got = run(graph(m, k, n, dtype, mode), np.ascontiguousarray(a.T) if mode == "t" else a,
              np.ascontiguousarray(b.T) if mode == "t" else b)
    with np.errstate(invalid="ignore"):
        e = (-a if mode == "f" else a).astype(np.float64) @ (b + b if mode == "f" else b).astype(np.float64)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(e))
    np.testing.assert_array_equal(np.where(np.isinf(e), got, 0), np.where(np.isinf(e), e, 0))
    assert np.isfinite(got[np.isfinite(e)]).all()
