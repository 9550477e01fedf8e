"""f32 products that a sum of products rounded once a term cannot get wrong:
one non-zero term a sum is the product rounded to nearest, whole numbers are
whole, and a sum that is zero is +0 as the interpreter's is, at large grids
of whole and of ragged tiles, at small ones and where k is split."""

import numpy as np
import pytest

from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.ir import F32, Graph

pytestmark = pytest.mark.gpu

# 210 tiles of 128x128, whole and ragged; 64x64 tiles; k in parts from 384
SIZES = [(1920, 1792), (1901, 1750), (300, 260), (64, 130)]


def product(a, b, mode):
    (m, k), n = a.shape, b.shape[1]
    if mode == "t":
        x, y = D.transpose(D.param("a", F32, (k, m))), D.transpose(D.param("b", F32, (n, k)))
        a, b = np.ascontiguousarray(a.T), np.ascontiguousarray(b.T)
    else:
        x, y = D.param("a", F32, (m, k)), D.param("b", F32, (k, n))
    c = H.compile(Graph.create("mm", [("c", D.matmul(x, y))]))
    try:
        return dict(H.run(c, [("a", a), ("b", b)]))["c"]
    finally:
        c.release()


@pytest.mark.parametrize("mode", ["d", "t"])
@pytest.mark.parametrize("k", [64, 256, 300, 1024])
@pytest.mark.parametrize("m,n", SIZES)
def test_one_term_a_sum(device, m, k, n, mode):
    r = np.random.default_rng(m + k)
    d, i = r.standard_normal(m).astype(np.float32), np.arange(m)
    d[::5] = 0  # rows of zeros
    a, b = np.zeros((m, k), np.float32), r.standard_normal((k, n)).astype(np.float32)
    a[i, i * 7 % k] = d
    e = d[:, None] * b[i * 7 % k]
    got = product(a, b, mode)
    np.testing.assert_array_equal(got, e)
    assert not np.signbit(got[e == 0]).any()


@pytest.mark.parametrize("mode", ["d", "t"])
@pytest.mark.parametrize("k", [64, 256, 300, 1024])
@pytest.mark.parametrize("m,n", SIZES)
def test_whole_numbers_that_cancel(device, m, k, n, mode):
    r = np.random.default_rng(n + k)
    a = r.integers(-3, 4, (m, k)).astype(np.float32)
    a[:, k // 2:2 * (k // 2)] = -a[:, :k // 2]
    b = r.integers(-3, 4, (k, n)).astype(np.float32)
    b[k // 2:2 * (k // 2), ::2] = b[:k // 2, ::2]  # every other column sums to zero
    b[2 * (k // 2):] = 0
    got = product(a, b, mode)
    e = a.astype(np.float64) @ b.astype(np.float64)
    np.testing.assert_array_equal(got, e)
    assert not np.signbit(got[e == 0]).any()
