"""Products that a sum of products rounded once a term cannot get wrong:
one non-zero term a sum is the product rounded to nearest, whole numbers are
whole, and a sum that is zero is +0 as the interpreter's is, in f32 and f64,
at large grids of whole and of ragged tiles, at small ones and where k is
split."""

import numpy as np
import pytest

from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.ir import F32, F64, Graph

pytestmark = pytest.mark.gpu

# f32: 210 tiles of 128x128, whole and ragged; 64x64 tiles; k in parts from
# 384. f64: 378 tiles of 64x64, k in two from 768; 32x32 tiles; k in parts.
SIZES = [(F32, 1920, 1792), (F32, 1901, 1750), (F32, 300, 260), (F32, 64, 130), (F64, 1300, 1100), (F64, 300, 260), (F64, 64, 130)]


def product(a, b, mode):
    (m, k), n, dtype = a.shape, b.shape[1], F32 if a.dtype == np.float32 else F64
    if mode == "t":
        x, y = D.transpose(D.param("a", dtype, (k, m))), D.transpose(D.param("b", dtype, (n, k)))
        a, b = np.ascontiguousarray(a.T), np.ascontiguousarray(b.T)
    else:
        x, y = D.param("a", dtype, (m, k)), D.param("b", dtype, (k, n))
    c = H.compile(Graph.create("mm", [("c", D.matmul(x, y))]))
    try:
        return dict(H.run(c, [("a", a), ("b", b)]))["c"]
    finally:
        c.release()


@pytest.mark.parametrize("mode", ["d", "t"])
@pytest.mark.parametrize("k", [64, 256, 300, 1024])
@pytest.mark.parametrize("dtype,m,n", SIZES)
def test_one_term_a_sum(device, dtype, m, k, n, mode):
    r = np.random.default_rng(m + k)
    d, i = r.standard_normal(m).astype(dtype.np), np.arange(m)
    d[::5] = 0  # rows of zeros
    a, b = np.zeros((m, k), dtype.np), r.standard_normal((k, n)).astype(dtype.np)
    a[i, i * 7 % k] = d
    e = d[:, None] * b[i * 7 % k]
    got = product(a, b, mode)
    np.testing.assert_array_equal(got, e)
    assert not np.signbit(got[e == 0]).any()


@pytest.mark.parametrize("mode", ["d", "t"])
@pytest.mark.parametrize("k", [64, 256, 300, 1024])
@pytest.mark.parametrize("dtype,m,n", SIZES)
def test_whole_numbers_that_cancel(device, dtype, m, k, n, mode):
    r = np.random.default_rng(n + k)
    a = r.integers(-3, 4, (m, k)).astype(dtype.np)
    a[:, k // 2:2 * (k // 2)] = -a[:, :k // 2]
    b = r.integers(-3, 4, (k, n)).astype(dtype.np)
    b[k // 2:2 * (k // 2), ::2] = b[:k // 2, ::2]  # every other column sums to zero
    b[2 * (k // 2):] = 0
    got = product(a, b, mode)
    e = a.astype(np.float64) @ b.astype(np.float64)
    np.testing.assert_array_equal(got, e)
    assert not np.signbit(got[e == 0]).any()
