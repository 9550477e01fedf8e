"""Float prefix sums over many small tiles are as close as few roundings can
be: the error of whole scans of positive values against that of rounding the
exact sums once."""

import numpy as np
import pytest

from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.ir import F32, F64, Graph

pytestmark = pytest.mark.gpu


# Chains of up to 256 tiles round a prefix where it is published, where it is
# read and where it joins an element: sqrt(3) roundings. Long chains round it
# once a hop; their bound lies between what carried prefixes (3.1) and plain
# ones (5.7) measure.
@pytest.mark.parametrize("dtype,shape,seeds,most", [(F32, (900_001,), 24, 1.75), (F64, (900_001,), 24, 1.75),
                                                    (F32, (30, 60_000), 8, 1.75), (F64, (1 << 25,), 5, 4.5)], ids=str)
def test_error_of_sums(device, dtype, shape, seeds, most):
    wide = np.float64 if dtype is F32 else np.longdouble
    x = D.param("x", dtype, shape)
    c = H.compile(Graph.create("s", [("p", (D.scan if len(shape) == 1 else D.scan_rows)(D.add, D.const(dtype, 0), x))]))
    err = once = 0.0
    try:
        for seed in range(seeds):
            v = np.random.default_rng(seed).random(shape).astype(dtype.np)
            e = np.cumsum(v.astype(wide), axis=-1)
            got = dict(H.run(c, [("x", v)]))["p"]
            err += float(((got - e) ** 2).sum() / (e ** 2).sum())
            once += float(((e.astype(dtype.np) - e) ** 2).sum() / (e ** 2).sum())
    finally:
        c.release()
    assert np.sqrt(err / once) <= most


@pytest.mark.parametrize("dtype", [F32, F64], ids=lambda d: d.name)
@pytest.mark.parametrize("n", [300_000, 3_000_000])
def test_zeros_infinities_and_nan(device, dtype, n):
    """A sum that overflows stays infinite, infinities of both signs give NaN
    from there on, and -0 stays -0 from an initial -0."""
    def scan(init, v):
        c = H.compile(Graph.create("s", [("p", D.scan(D.add, D.const(dtype, init), D.param("x", dtype, (n,))))]))
        try:
            return dict(H.run(c, [("x", v)]))["p"]
        finally:
            c.release()

    v = np.full(n, -0.0, dtype.np)
    assert np.signbit(scan(-0.0, v)).all()
    assert not np.signbit(scan(0.0, v)).any()
    v = np.ones(n, dtype.np)
    v[n // 3] = np.inf
    got = scan(0, v)
    np.testing.assert_array_equal(got[: n // 3], np.arange(1, n // 3 + 1))
    assert (got[n // 3:] == np.inf).all()
    v[n // 2] = -np.inf
    got = scan(0, v)
    assert (got[n // 3:n // 2] == np.inf).all() and np.isnan(got[n // 2:]).all()
    big = np.finfo(dtype.np).max
    v = np.zeros(n, dtype.np)
    v[[5, n // 2]] = big
    got = scan(0, v)
    assert (got[5:n // 2] == big).all() and (got[n // 2:] == np.inf).all()
