"""Matrix products of few tiles, whose k is split over workgroups: whole and
ragged slices of k, every operand mode, both dtypes, up to the most slices,
against the exact product and against the unsplit kernel; and the products
that go without for the scratch they would take."""

import numpy as np
import pytest

from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.ir import F32, F64, I32, Graph


def graph(dtype, m, k, n, mode):
    if mode == "t":
        a, b = D.transpose(D.param("a", dtype, (k, m))), D.transpose(D.param("b", dtype, (n, k)))
    else:
        a, b = D.param("a", dtype, (m, k)), D.param("b", dtype, (k, n))
    if mode == "f":
        a, b = D.map(D.neg, a), D.map(lambda v: D.add(v, v), b)
    return Graph.create("mm", [("c", D.matmul(a, b))])


def roles(g):
    return [line.split()[2] for line in H.plan(g).splitlines() if line.startswith("kernel")]


def run(g, ins, monkeypatch, knobs):
    monkeypatch.setenv("CCHIP_TUNE", knobs)
    c = H.compile(g)
    try:
        return dict(H.run(c, ins))["c"]
    finally:
        c.release()


SIZES = [(64, 1024, 64), (33, 1025, 65), (64, 1023, 100), (200, 2000, 96), (300, 1500, 310), (40, 20001, 40)]


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["d", "t", "f"])
@pytest.mark.parametrize("dtype,m,k,n", [(d, *s) for s in SIZES for d in (F32, F64)] + [(F32, 700, 901, 700), (F64, 1300, 800, 1100)])
def test_split_k(device, monkeypatch, dtype, m, k, n, mode):
    rng = np.random.default_rng(m + k + n)
    a, b = rng.standard_normal((m, k)).astype(dtype.np), rng.standard_normal((k, n)).astype(dtype.np)
    g = graph(dtype, m, k, n, mode)
    assert len(roles(g)) == 2 and roles(g)[1] == "matmul_ksum"
    ins = [("a", np.ascontiguousarray(a.T) if mode == "t" else a), ("b", np.ascontiguousarray(b.T) if mode == "t" else b)]
    got, one = run(g, ins, monkeypatch, ""), run(g, ins, monkeypatch, "mm_ksplit=0")
    assert len(roles(g)) == 1
    x, y = (-a, b + b) if mode == "f" else (a, b)
    # k rounded steps each, in either order; the f64 product itself is
    # rounded as often
    u = 2.0 ** -24 if dtype is F32 else 2.0 ** -52
    bound = (k + 40) * u * (np.abs(x).astype(np.float64) @ np.abs(y).astype(np.float64))
    e = x.astype(np.float64) @ y.astype(np.float64)
    assert (np.abs(got - e) <= bound).all() and (np.abs(one - e) <= bound).all()
    # whole numbers: every partial sum is exact
    ins = [(name, np.rint(v * 2).astype(dtype.np)) for name, v in ins]
    np.testing.assert_array_equal(run(g, ins, monkeypatch, ""), run(g, ins, monkeypatch, "mm_ksplit=0"))


def test_partial_products_leave_the_allocation_free_scratch_its_room():
    """A program within 32 MiB of scratch without the partial products, and
    not with them, goes without; one beyond it either way splits."""
    x, y = D.param("x", F32, (256, 2048)), D.param("y", F32, (2048, 256))
    c = D.matmul(x, y)
    assert len(roles(Graph.create("one", [("c", c)]))) == 2

    def scratch(g):
        return sum(int(line.split()[4]) * 4 for line in H.plan(g).splitlines() if line.startswith("buffer") and line.endswith("scratch"))

    seen = set()
    for n in range(1 << 18, 6 << 20, 1 << 16):
        s = D.scatter_add(D.param("i", I32, (n,)), D.param("v", F32, (n,)), (1 << 17,))
        split = "matmul_ksum" in roles(Graph.create("both", [("c", c), ("s", s)]))
        alone = scratch(Graph.create("s", [("s", s)]))
        both = alone + scratch(Graph.create("one", [("c", c)]))
        # a buffer's end is rounded up by less than 256 bytes, and up to 1 MiB
        # of small buffers is not counted
        if both < (32 << 20) - 4096 or alone > 33 << 20:
            assert split
        elif both > 33 << 20 and alone < 32 << 20:
            assert not split
        seen.add((split, alone > 33 << 20))
    assert seen == {(True, False), (False, False), (True, True)}
