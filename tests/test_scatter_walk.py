"""How a scatter_add's workgroups and waves share its tiles: no shape is left
with a few workgroups because their scratch gave way first, and a workgroup's
tiles are walked in as few turns of its waves as they need. The sums over
such shares, exactly, on the device."""

import re

import numpy as np
import pytest

from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.ir import F32, F64, I32, Graph


def graph(dtype, n, bins):
    return Graph.create("s", [("h", D.scatter_add(D.param("i", I32, (n,)), D.param("v", dtype, (n,)), (bins,)))])


def grids(g):
    return {line.split()[2]: int(line.split()[4]) for line in H.plan(g).splitlines() if line.startswith("kernel")}


@pytest.mark.parametrize("dtype,n,bins,least", [(F64, 60_000_000, 100_000, 200), (F64, 20_000_000, 1_000_000, 400),
                                                (F64, 20_000_000, 30_000, 90), (F32, 300_000, 60_000, 60),
                                                (F64, 300_000, 30_000, 64)])
def test_workgroups_of_the_accumulate(dtype, n, bins, least):
    assert grids(graph(dtype, n, bins))["scatter_accumulate"] >= least


@pytest.mark.parametrize("dtype,n,bins", [(F32, 100_000, 100_000), (F32, 300_000, 30_000), (F64, 100_000, 60_000)])
def test_few_tiles_are_walked_in_one_turn(dtype, n, bins):
    g = graph(dtype, n, bins)
    k = grids(g)
    slices = -(-bins // 4096)
    tiles = -(-k["scatter_partition"] // (k["scatter_accumulate"] // slices))
    assert int(re.search(r"tb \+= (\d+)", H.source(g)).group(1)) >= tiles > 8


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, F64, I32], ids=lambda d: d.name)
@pytest.mark.parametrize("n,bins", [(20_011, 16_385), (99_991, 100_003), (99_991, 30_011), (450_001, 30_011), (450_001, 250_007),
                                    (1_000_003, 40_961), (3_000_017, 300_007), (5_000_011, 1_000_003)])
def test_sums_of_shared_tiles(device, dtype, n, bins):
    r = np.random.default_rng(n + bins)
    i = r.integers(0, bins, n).astype(np.int32)
    i[: n // 7] = r.integers(0, 64, n // 7)  # runs of very different lengths
    v = r.integers(-3, 4, n).astype(dtype.np)  # every partial sum is exact
    idx = D.param("i", I32, (n,))
    h = D.scatter_add(idx, D.param("v", dtype, (n,)), (bins,))
    c = H.compile(Graph.create("s", [("h", h), ("back", D.gather(idx, h))]))
    try:
        got = dict(H.run(c, [("i", i), ("v", v)]))
    finally:
        c.release()
    e = np.bincount(i, v.astype(np.float64), bins).astype(dtype.np)
    np.testing.assert_array_equal(got["h"], e)
    np.testing.assert_array_equal(got["back"], e[i])
