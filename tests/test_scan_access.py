"""Which scans stream (non-temporal accesses), read off the generated source:
4-byte values beyond the MALL, and 8-byte ones only in the 2-element groups of
a whole-tensor scan; 4-element groups of 8-byte values are two interleaved
accesses, which stream at a fraction of the plain rate."""

import pytest

from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.ir import F32, F64, I64, Graph


def streamed(dtype, shape):
    x = D.param("x", dtype, shape)
    f = D.scan if len(shape) == 1 else D.scan_rows
    g = Graph.create("s", [("p", f(D.add, D.const(dtype, 0), x))])
    body = H.source(g).split('extern "C"', 1)[1]
    return any(t in body for t in ("nt(b", "cc_bst4<float, 2>", "_nt<"))


@pytest.mark.parametrize("dtype,shape,yes", [
    (F64, (5000, 8192), False), (F64, (3000, 12001), False),  # one tile a row, whole and odd groups
    (F64, (1000, 17000), False), (I64, (500, 80001), False),  # several
    (F64, (1 << 27,), True), (I64, ((1 << 27) + 1,), True),
    (F32, (5000, 16384), True), (F32, (1000, 80000), True), (F32, (1 << 28,), True),
    (F64, (1000, 8192), False), (F32, (1000, 8192), False),  # in the MALL
], ids=str)
def test_scans_that_stream(dtype, shape, yes):
    assert streamed(dtype, shape) == yes
