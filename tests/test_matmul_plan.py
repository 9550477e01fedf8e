"""Where products split k: f64 ones of 64x64 tiles in two, and which programs
go without for the room their partial products take."""

import pytest

from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd.examples import configs as C
from cudacaml_amd.ir import F32, F64, I32, Graph


@pytest.mark.parametrize("m,n,k,parts", [(1300, 1100, 800, 2), (1536, 1024, 800, 2), (1536, 1024, 767, 1), (1280, 1280, 800, 1),
                                         (1280, 1280, 1200, 1), (1344, 1344, 1599, 1), (1280, 1280, 1600, 2),
                                         (1500, 1101, 2001, 2), (1408, 1344, 4000, 1)])
def test_parts_of_k(m, n, k, parts):
    kernels = [line.split() for line in H.plan(C.matmul(n, F64, k=k, m=m)).splitlines() if line.startswith("kernel")]
    tiles = -(-m // 64) * -(-n // 64)
    assert int(kernels[0][4]) == parts * tiles and len(kernels) == parts


def test_parts_of_k_give_way_to_the_allocation_free_scratch(monkeypatch):
    """A program splits k unless its scratch counts for more than 32 MiB with
    the partial products and for at most that without; buffers of up to 256
    KiB count from their 1 MiB on."""
    cap, size = 32 << 20, {"f32": 4, "f64": 8, "i32": 4, "i64": 8}

    def counted(plan):
        room = [-(-int(f[4]) * size[f[3]] // 256) * 256 for f in map(str.split, plan.splitlines())
                if f[:1] == ["buffer"] and f[-1] == "scratch"]
        return 256 + sum(room) - min(1 << 20, sum(r for r in room if r <= 256 << 10))

    c = D.matmul(D.param("x", F32, (256, 2048)), D.param("y", F32, (2048, 256)))
    seen = set()
    for scans in (0, 4):  # about 175 KiB of tile words each
        words = [("p%d" % i, D.scan(D.add, D.const(F64, 0), D.param("d%d" % i, F64, (1 << 27,)))) for i in range(scans)]
        for n in range(15 << 17, 34 << 17, 9999):
            s = D.scatter_add(D.param("i", I32, (n,)), D.param("v", F32, (n,)), (1 << 17,))
            g = Graph.create("g", [("c", c), ("s", s)] + words)
            monkeypatch.setenv("CCHIP_TUNE", "mm_ksplit=0")
            without = counted(H.plan(g))
            monkeypatch.delenv("CCHIP_TUNE")
            plan = H.plan(g)
            split = "matmul_ksum" in plan
            extra = 16 * 256 * 256 * 4
            assert split == (without + extra <= cap or without > cap)
            assert counted(plan) == without + (extra if split else 0)
            seen.add((split, without > cap, scans))
    assert len(seen) == 6
