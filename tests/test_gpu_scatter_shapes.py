"""scatter_add with gather back over the shapes its launch rules divide:
slices of 4096 to 16384 bins, sums of few and of many partial tables, both
partition tiles, and the gather read plainly or back through the
partition. Integers bit for bit against numpy, floats within the bound of
any order of a bin's additions, back exactly h[idx]."""

import numpy as np
import pytest

from cudacaml_amd import backend_hip as H
from cudacaml_amd.examples import configs as C
from cudacaml_amd.ir import F32, F64, I32

pytestmark = pytest.mark.gpu

# (values, bins): one slice with 2 to 600 partial tables; several slices at
# the edges of a slice and of the rule for their size; few slices with many
# workgroups each; both sides of the lines of the tile and the plain gather
SHAPES = [(16384, 100), (140000, 1000), (500003, 8191), (5000011, 3000), (300001, 16385), (300001, 64 * 4096),
          (300001, 64 * 4096 + 1), (3000007, 20000), ((2 << 20) + 1, 65536), ((2 << 20) + 1, 65537),
          ((8 << 20) + 9, 50000), ((2 << 20) + 3, (1 << 19) + 1)]


@pytest.mark.parametrize("dtype", [F32, F64, I32], ids=lambda d: d.name)
@pytest.mark.parametrize("n,bins", SHAPES)
def test_scatter_shapes(device, dtype, n, bins):
    r = np.random.default_rng(n + bins)
    idx = r.integers(0, bins, n).astype(np.int32)
    idx[::11] = idx[0]  # a crowded bin
    src = r.integers(-1000, 1000, n).astype(np.int32) if dtype is I32 else r.standard_normal(n).astype(dtype.np)
    c = H.compile(C.scatter_gather(n, bins, dtype))
    try:
        got = dict(H.run(c, [("idx", idx), ("src", src)]))
    finally:
        c.release()
    h = got["h"]
    np.testing.assert_array_equal(got["back"], h[idx])
    if dtype is I32:
        e = np.bincount(idx, src.astype(np.float64), bins)  # exact below 2^53
        np.testing.assert_array_equal(h.astype(np.int64), e.astype(np.int64))
    else:
        e = np.bincount(idx, src.astype(np.float64), bins)
        s, m = np.bincount(idx, np.abs(src.astype(np.float64)), bins), np.bincount(idx, minlength=bins)
        # m additions in any order, and as many in the float64 reference
        u = 2.0 ** -24 if dtype is F32 else 2.0 ** -52
        assert (np.abs(h - e) <= m * u * s).all()
