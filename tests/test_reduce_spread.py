"""How many workgroups a reduction of a long element function takes: one of
256 elements each where a row gives too few of 4096, up to 2048 in all, and
4096 each beyond."""

import pytest

from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.ir import F32, F64, Graph


@pytest.mark.parametrize("dtype", [F32, F64], ids=lambda d: d.name)
@pytest.mark.parametrize("shape,groups", [((30_000,), 118), ((500_000,), 1954), (((3 << 18) - 1,), 1536), (((3 << 18),), 192), ((1 << 20,), 256), ((2_000_000,), 489),
                                          ((4_000_000,), 977), ((3, 30_000), 354), ((4, 1 << 20), 1024)], ids=str)
def test_workgroups_of_a_long_function(dtype, shape, groups):
    m = D.param("x", dtype, shape)
    for i in range(24):
        m = D.map(lambda v, i=i: D.add(D.mul(v, D.const(dtype, 0.5)), D.const(dtype, i / 64)), m)
    r = D.reduce if len(shape) == 1 else D.reduce_rows
    plan = H.plan(Graph.create("h", [("s", r(D.add, D.const(dtype, 0), D.map(D.exp, m)))]))
    assert {line.split()[2]: int(line.split()[4]) for line in plan.splitlines() if line.startswith("kernel")}["reduce_split"] == groups
