"""f32 products through three bf16 planes an operand: every operand mode at
whole and ragged tiles, within the bound of a sum of K rounded steps; and
the tiles that meet a value the planes cannot hold (an infinity, a NaN, a
value past 2^60 or below 2^-100), which take the f32 instructions and keep
their results."""

import numpy as np
import pytest

from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.ir import F32, Graph

pytestmark = pytest.mark.gpu


def graph(m, k, n, mode):
    if mode == "t":
        a, b = D.transpose(D.param("a", F32, (k, m))), D.transpose(D.param("b", F32, (n, k)))
    else:
        a, b = D.param("a", F32, (m, k)), D.param("b", F32, (k, n))
    if mode == "f":
        a, b = D.map(D.neg, a), D.map(lambda v: D.add(v, v), b)
    return Graph.create("mm", [("c", D.matmul(a, b))])


def run(monkeypatch, knobs, g, a, b, mode):
    monkeypatch.setenv("CCHIP_TUNE", knobs)
    assert ("cc_split4" in H.source(g)) == ("mm_split=2" in knobs)
    c = H.compile(g)
    try:
        if mode == "t":
            a, b = np.ascontiguousarray(a.T), np.ascontiguousarray(b.T)
        return dict(H.run(c, [("a", a), ("b", b)]))["c"]
    finally:
        c.release()


def exact(a, b, mode):
    """The operands as the program rounds them, in float64."""
    with np.errstate(over="ignore"):
        a, b = (-a, b + b) if mode == "f" else (a, b)
    return a.astype(np.float64), b.astype(np.float64)


SIZES = [(128, 64, 128), (128, 96, 256), (129, 65, 127), (127, 100, 130), (256, 288, 128), (131, 545, 257), (200, 1024, 200)]


@pytest.mark.parametrize("mode", ["d", "t", "f"])
@pytest.mark.parametrize("m,k,n", SIZES)
@pytest.mark.parametrize("spread", [0, 30])
def test_split_product(device, monkeypatch, m, k, n, mode, spread):
    rng = np.random.default_rng(m + 1000 * k + n)
    a, b = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    if spread:  # magnitudes over 2 * spread octaves, and zeros of both signs
        a, b = a * 2.0 ** rng.uniform(-spread, spread, a.shape), b * 2.0 ** rng.uniform(-spread, spread, b.shape)
        a[rng.random(a.shape) < 0.1], b[rng.random(b.shape) < 0.1] = 0.0, -0.0
    a, b = a.astype(np.float32), b.astype(np.float32)
    got = run(monkeypatch, "mm_split=2", graph(m, k, n, mode), a, b, mode)
    aw, bw = exact(a, b, mode)
    # 12 roundings of the accumulator for 16 steps and one a chunk, each at
    # most u times the partial sums' bound, and 2^-23 |x y| a product for
    # what the planes leave out
    bound = (k + 4) * 2.0 ** -24 * (np.abs(aw) @ np.abs(bw))
    assert (np.abs(got - aw @ bw) <= bound).all()


ODD = [np.inf, -np.inf, np.nan, np.float32(1e30), -np.float32(2.0 ** 60), np.float32(1e-31), np.float32(1e-38), np.float32(1e-45),
       np.float32(1e37)]


@pytest.mark.parametrize("mode", ["d", "t", "f"])
@pytest.mark.parametrize("value", ODD, ids=str)
@pytest.mark.parametrize("where", ["a", "b", "both"])
def test_values_outside_the_planes_take_the_f32_instructions(device, monkeypatch, value, where, mode):
    m, k, n = 300, 300, 260
    rng = np.random.default_rng(5)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    if where != "b":
        a[140, k - 1] = value  # the second tile row, in the last k tile
    if where != "a":
        b[3, 258] = value  # the third tile column, in the first
    g = graph(m, k, n, mode)
    got = run(monkeypatch, "mm_split=2", g, a, b, mode)
    f32 = run(monkeypatch, "mm_split=0", g, a, b, mode)
    hit = np.zeros((m, n), bool)
    if where != "b":
        hit[128:256] = True
    if where != "a":
        hit[:, 256:] = True
    aw, bw = exact(a, b, mode)
    with np.errstate(invalid="ignore", over="ignore"):
        e = (aw @ bw).astype(np.float32)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(e))
    np.testing.assert_array_equal(got[np.isinf(e)], e[np.isinf(e)])
    # the f32 instructions on those tiles, in another tile size
    both = hit & np.isfinite(e)
    scale = np.abs(np.nan_to_num(aw, posinf=0, neginf=0)) @ np.abs(np.nan_to_num(bw, posinf=0, neginf=0))
    assert (np.abs(got[both].astype(np.float64) - f32[both]) <= (k + 4) * 2.0 ** -23 * scale[both]).all()
    rest = ~hit & np.isfinite(e)
    assert (np.abs(got[rest] - e.astype(np.float64)[rest]) <= (k + 5) * 2.0 ** -24 * scale[rest]).all()


def test_a_tile_of_tiny_values_keeps_its_precision(device, monkeypatch):
    """Every operand value near 2^-110, times values near 2^50: 24 bits of
    each count."""
    rng = np.random.default_rng(6)
    a = (rng.standard_normal((128, 128)) * 2.0 ** -112).astype(np.float32)
    b = (rng.standard_normal((128, 128)) * 2.0 ** 50).astype(np.float32)
    got = run(monkeypatch, "mm_split=2", graph(128, 128, 128, "d"), a, b, "d").astype(np.float64)
    aw, bw = exact(a, b, "d")
    assert (np.abs(got - aw @ bw) <= 132 * 2.0 ** -24 * (np.abs(aw) @ np.abs(bw))).all()


def test_large_grids_take_the_planes(device):
    assert "cc_split4" in H.source(graph(2048, 64, 2048, "d"))
    assert "cc_split4" not in H.source(graph(1024, 1024, 1024, "d"))
    assert "cc_split4" not in H.source(graph(2048, 48, 2048, "d"))


@pytest.mark.parametrize("k", [64, 256, 288, 300, 1024])
def test_no_mean_error(device, monkeypatch, k):
    """The bf16 instructions cut towards minus infinity; the flipped tiles
    take the mean of it away. The mean of m n independent errors of root
    mean square e is within 6 e / sqrt(m n); a whole tile's cut left over
    would be 3e-9 of the result's root mean square or more, 20 times that."""
    m = n = 1024
    rng = np.random.default_rng(k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    err = run(monkeypatch, "mm_split=2", graph(m, k, n, "d"), a, b, "d") - a.astype(np.float64) @ b.astype(np.float64)
    assert abs(err.mean()) <= 6 * err.std() / np.sqrt(m * n)
