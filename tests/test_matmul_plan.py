"""Where f64 products of 64x64 tiles split k in two: while twice the tiles
are three a CU, and beyond that for long k alone."""

import pytest

from cudacaml_amd import backend_hip as H
from cudacaml_amd.examples import configs as C
from cudacaml_amd.ir import F64


@pytest.mark.parametrize("m,n,k,parts", [(1300, 1100, 800, 2), (1536, 1024, 800, 2), (1536, 1024, 767, 1), (1280, 1280, 800, 1),
                                         (1280, 1280, 1200, 1), (1344, 1344, 1599, 1), (1280, 1280, 1600, 2),
                                         (1500, 1101, 2001, 2), (1408, 1344, 4000, 1)])
def test_parts_of_k(m, n, k, parts):
    kernels = [line.split() for line in H.plan(C.matmul(n, F64, k=k, m=m)).splitlines() if line.startswith("kernel")]
    tiles = -(-m // 64) * -(-n // 64)
    assert int(kernels[0][4]) == parts * tiles and len(kernels) == parts
