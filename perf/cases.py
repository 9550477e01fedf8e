"""What is timed when the backend's speed is measured: the array programs a
user of the DSL compiles once and runs many times, through
``backend_hip.compile`` and ``run_resident_into`` (inputs and outputs resident
on the GPU) or ``backend_hip.run`` (host values in, host values out).

The programs are those of ``cudacaml_amd/examples`` and of the benchmark, at
its sizes and at odd ones: element-wise maps with a sum, row folds and row
scans, whole-tensor scans, scatter_add with its gather back, matrix products
alone and in a gradient, and the Monte Carlo pricers.
"""

import math

import torch

from cudacaml_amd import backend_hip as H
from cudacaml_amd import dsl as D
from cudacaml_amd import grad as G
from cudacaml_amd.examples import black_scholes as bs
from cudacaml_amd.examples import configs as C
from cudacaml_amd.examples import saxpy as sx
from cudacaml_amd.ir import F32, F64, I32, I64, Graph
from cudacaml_amd.runtime import Buffer

DTYPES = {"f32": F32, "f64": F64, "i32": I32, "i64": I64}
TORCH = {F32: torch.float32, F64: torch.float64, I32: torch.int32, I64: torch.int64}
SIZE = {"f32": 4, "f64": 8, "i32": 4, "i64": 8}
DEV = "cuda"


def listed():
    return [
        # One quote from a pricing service: host scalars in, a price out. What
        # counts is latency: an upload, a few launches, a download.
        {"name": "price_100k_f32", "kind": "price", "paths": 100_000, "dtype": "f32"},
        # The first program everybody writes, in double precision, on a length
        # that is no power of two: r = 2x + y and the sum of r.
        {"name": "saxpy_30M_f64", "kind": "saxpy", "n": 30_000_001, "dtype": "f64"},
        # The benchmark's row workload: sum, max and running sum of each row.
        {"name": "rows_8192x8192_f32", "kind": "rows", "rows": 8192, "cols": 8192, "dtype": "f32"},
        # The same on a table of odd shape, a few thousand records wide.
        {"name": "rows_1500x3001_f64", "kind": "rows", "rows": 1500, "cols": 3001, "dtype": "f64"},
        # The benchmark's prefix sum, the largest tensor of the list.
        {"name": "scan_2p28_i32", "kind": "scan", "n": 1 << 28, "dtype": "i32"},
        # A cumulative sum of ten million doubles.
        {"name": "scan_10M_f64", "kind": "scan", "n": 10_000_019, "dtype": "f64"},
        # The benchmark's histogram with weights, and each value's bin total.
        {"name": "scatter_2p26_f32", "kind": "scatter", "n": 1 << 26, "bins": 1 << 20, "dtype": "f32"},
        # Counting five million events into a table of odd size.
        {"name": "scatter_5M_i32", "kind": "scatter", "n": 5_000_011, "bins": 100_003, "dtype": "i32"},
        # The benchmark's matrix product.
        {"name": "matmul_4096_f32", "kind": "matmul", "m": 4096, "n": 4096, "k": 4096, "dtype": "f32"},
        # A double-precision product of three different, odd sides.
        {"name": "matmul_1500x1101x2001_f64", "kind": "matmul", "m": 1500, "n": 1101, "k": 2001, "dtype": "f64"},
        # One training step of a linear layer under squared error, forward and
        # backward: the loss and both gradients, a batch of 1500.
        {"name": "lsq_1500x700x901_f32", "kind": "lsq", "m": 1500, "n": 901, "k": 700, "dtype": "f32"},
        # The 64-step pricer with its pathwise delta and vega: the whole of the
        # engine in one graph, forward and backward.
        {"name": "greeks_2p18x64_f64", "kind": "greeks", "paths": 1 << 18, "steps": 64, "dtype": "f64"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["price", "saxpy", "rows", "scan", "scatter", "matmul", "matmul", "lsq", "greeks"])
    f = rng.choice(["f32", "f64"])
    if kind == "price":
        return {"kind": kind, "paths": _log(rng, 1000, 1 << 22), "dtype": f}
    if kind == "saxpy":
        return {"kind": kind, "n": _log(rng, 1000, 1 << 27), "dtype": f}
    if kind == "rows":
        cols = _log(rng, 32, 1 << 16)
        return {"kind": kind, "rows": max(1, min(_log(rng, 8, 1 << 16), (1 << 26) // cols)), "cols": cols, "dtype": f}
    if kind == "scan":
        d = rng.choice(["i32", "i64", "f32", "f64"])
        return {"kind": kind, "n": _log(rng, 1000, 1 << (28 if SIZE[d] == 4 else 27)), "dtype": d}
    if kind == "scatter":
        n = _log(rng, 10_000, 1 << 26)
        return {"kind": kind, "n": n, "bins": _log(rng, 100, min(n, 1 << 21)), "dtype": rng.choice(["f32", "f64", "i32"])}
    if kind in ("matmul", "lsq"):
        side = 4096 if f == "f32" else 2048
        if kind == "lsq":  # three products
            side //= 2
        return {"kind": kind, "m": _log(rng, 64, side), "n": _log(rng, 64, side), "k": _log(rng, 64, side), "dtype": f}
    # In f32 a draw of the inverse CDF is infinite with probability 2^-24.4
    # (the uniform rounds to 0 or 1), so f32 paths stay short of that.
    steps = rng.choice([16, 50, 64, 100])
    return {"kind": kind, "paths": _log(rng, 1000, (1 << (22 if f == "f32" else 26)) // steps), "steps": steps, "dtype": f}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _philox(key, n, start=0):
    """Word 0 of Philox-4x32-10 at counters (i, 0, 0, 0), key (key, 0), as
    int64 in [0, 2^32): the stream of ``Rng.u32``. 64-bit products wrap, and
    their low 64 bits are what the words are cut from."""
    m = 0xFFFFFFFF
    c0 = torch.arange(start, start + n, dtype=torch.int64, device=DEV) & m
    c1, c2, c3 = torch.zeros_like(c0), torch.zeros_like(c0), torch.zeros_like(c0)
    k0, k1 = key & m, 0
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = ((p1 >> 32) & m) ^ c1 ^ k0, p1 & m, ((p0 >> 32) & m) ^ c3 ^ k1, p0 & m
        k0, k1 = (k0 + 0x9E3779B9) & m, (k1 + 0xBB67AE85) & m
    return c0


def _key(case, seed):
    """The Philox key of a pricer. In f32 the 128 largest and the 64 smallest
    words give an infinite normal draw, and so an infinite price: the first
    key after the seed's own that meets none of them is taken."""
    key = 1 + 1000 * (int(seed) % 1_000_000)
    if case["dtype"] == "f32":
        n = case["paths"] * case.get("steps", 1)
        while True:
            w = _philox(key, n)
            if int(w.max()) < 2 ** 32 - 128 and int(w.min()) >= 64:
                break
            key += 1
    return key


def _arrays(case, seed):
    """The program's tensors by name, drawn on the GPU."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    d = TORCH[DTYPES[case["dtype"]]]
    kind = case["kind"]

    def uniform(shape, lo, hi):
        return torch.empty(shape, dtype=d, device=DEV).uniform_(lo, hi, generator=g)

    def normal(shape):
        return torch.empty(shape, dtype=d, device=DEV).normal_(generator=g)

    def ints(shape, hi, dtype):
        return torch.randint(0, hi, shape, dtype=dtype, device=DEV, generator=g)

    if kind == "saxpy":
        return {"x": uniform((case["n"],), 0, 1), "y": uniform((case["n"],), 0, 1)}
    if kind == "rows":
        return {"x": uniform((case["rows"], case["cols"]), 0, 1)}
    if kind == "scan":
        n = (case["n"],)
        return {"v": ints(n, 16, d) if case["dtype"][0] == "i" else uniform(n, 0, 1)}
    if kind == "scatter":
        n = (case["n"],)
        src = ints(n, 16, d) if case["dtype"][0] == "i" else uniform(n, 0, 1)
        return {"idx": ints(n, case["bins"], torch.int32), "src": src}
    if kind == "matmul":
        return {"a": normal((case["m"], case["k"])), "b": normal((case["k"], case["n"]))}
    if kind == "lsq":
        return {"x": normal((case["m"], case["k"])), "w": normal((case["k"], case["n"])),
                "y": normal((case["m"], case["n"]))}
    m = bs.market
    out = {k: torch.tensor(v, dtype=d, device=DEV) for k, v in (("s0", m.s0), ("vol", m.vol), ("rate", m.rate))}
    out["seed"] = torch.tensor(_key(case, seed), dtype=torch.int32, device=DEV)
    return out


def _graph(case):
    kind, d = case["kind"], DTYPES[case["dtype"]]
    if kind == "price":
        return bs.call_mc(case["paths"], d)
    if kind == "saxpy":
        if d is F32:
            return sx.program(case["n"], 2.0)
        x, y = D.param("x", d, (case["n"],)), D.param("y", d, (case["n"],))
        r = D.map2(lambda a, b: D.add(D.mul(D.const(d, 2.0), a), b), x, y)
        return Graph.create("saxpy", [("r", r), ("s", D.reduce(D.add, D.const(d, 0.0), r))])
    if kind == "rows":
        return C.rows(case["rows"], case["cols"], d)
    if kind == "scan":
        v = D.param("v", d, (case["n"],))
        return Graph.create("scan", [("p", D.scan(D.add, D.const(d, 0 if d in (I32, I64) else 0.0), v))])
    if kind == "scatter":
        return C.scatter_gather(case["n"], case["bins"], d)
    if kind == "matmul":
        return C.matmul(case["n"], d, k=case["k"], m=case["m"])
    if kind == "lsq":
        m, n, k = case["m"], case["n"], case["k"]
        e = D.map2(D.sub, D.matmul(D.param("x", d, (m, k)), D.param("w", d, (k, n))), D.param("y", d, (m, n)))
        loss = D.reduce(D.add, D.const(d, 0.0), D.map(lambda v: D.mul(v, v), e))
        return G.grad(Graph.create("lsq", [("loss", loss)]), "loss", ["x", "w"])
    return bs.call_paths_greeks(case["paths"], case["steps"], d)


def _resident(t, dtype):
    return H.Resident(Buffer(t.data_ptr(), t.numel() * t.element_size()), dtype, tuple(t.shape))


def prepare(case, seed):
    arrays = _arrays(case, seed)
    c = H.compile(_graph(case))
    if case["kind"] == "price":
        return {"program": c, "host": {k: t.cpu().numpy() for k, t in arrays.items()}}
    outs = {o.name: torch.empty(o.shape, dtype=TORCH[o.dtype], device=DEV) for o in c.outputs}
    return {"program": c, "inputs": {p.name: _resident(arrays[p.name], p.dtype) for p in c.params},
            "outputs": {o.name: _resident(outs[o.name], o.dtype) for o in c.outputs},
            "tensors": (arrays, outs)}


def run(state):
    if "host" in state:
        return dict(H.run(state["program"], state["host"]))
    H.run_resident_into(state["program"], state["inputs"], state["outputs"], sync=False)
    return state["tensors"][1]


# ---------------------------------------------------------------------------
# What a pass cannot do without, and what it gives
# ---------------------------------------------------------------------------

# Operations of one normal draw: Philox's ten rounds (two wide products, four
# xors, two key additions each) and about twenty for the inverse CDF.
DRAW_OPS = 100


def work(case):
    kind, z = case["kind"], SIZE[case["dtype"]]
    if kind == "price":
        return {"bytes": 4 * z + 4, "flops": case["paths"] * (DRAW_OPS + 30)}
    if kind == "saxpy":
        return {"bytes": 3 * z * case["n"] + z, "flops": 3 * case["n"]}
    if kind == "rows":
        n = case["rows"] * case["cols"]
        return {"bytes": 2 * z * n + 2 * z * case["rows"], "flops": 3 * n}
    if kind == "scan":
        return {"bytes": 2 * z * case["n"], "flops": case["n"]}
    if kind == "scatter":
        return {"bytes": (4 + 2 * z) * case["n"] + z * case["bins"], "flops": case["n"]}
    if kind in ("matmul", "lsq"):
        m, n, k = case["m"], case["n"], case["k"]
        if kind == "matmul":
            return {"bytes": z * (m * k + k * n + m * n), "flops": 2 * m * n * k}
        return {"bytes": z * (2 * m * k + 2 * k * n + m * n + 1), "flops": 6 * m * n * k + 4 * m * n}
    return {"bytes": 6 * z + 4, "flops": case["paths"] * case["steps"] * (DRAW_OPS + 80)}


def tolerance(case):
    d, kind = case["dtype"], case["kind"]
    if d[0] == "i":
        return "exact"
    if kind in ("price", "greeks"):
        return {"rel": 2e-6 if d == "f32" else 2e-13}
    return {"rel": 4e-6 if d == "f32" else 5e-15}


def _normals(case, key):
    """The pricer's normal draws in 64 bits, 2^24 at a time."""
    steps = case.get("steps", 1)
    rows = max(1, (1 << 24) // steps)
    for lo in range(0, case["paths"], rows):
        hi = min(case["paths"], lo + rows)
        w = _philox(key, (hi - lo) * steps, lo * steps)
        u = (w.double() + 0.5) * 2.0 ** -32
        yield torch.special.ndtri(u).reshape(hi - lo, steps)


def exact(case, seed):
    kind = case["kind"]
    v = _arrays(case, seed)
    if kind == "saxpy":
        r = 2.0 * v["x"].double() + v["y"].double()
        return {"r": r, "s": r.sum()}
    if kind == "rows":
        x = v["x"].double()
        return {"sum": x.sum(1), "max": x.max(1).values, "scan": x.cumsum(1)}
    if kind == "scan":
        p = v["v"].to(torch.int64 if case["dtype"][0] == "i" else torch.float64).cumsum(0)
        return {"p": p.to(TORCH[DTYPES[case["dtype"]]]) if case["dtype"][0] == "i" else p}
    if kind == "scatter":
        wide = torch.int64 if case["dtype"][0] == "i" else torch.float64
        i = v["idx"].long()
        h = torch.zeros(case["bins"], dtype=wide, device=DEV).index_add_(0, i, v["src"].to(wide))
        h = h.to(torch.int32) if case["dtype"][0] == "i" else h
        return {"h": h, "back": h[i]}
    if kind == "matmul":
        return {"c": v["a"].double() @ v["b"].double()}
    if kind == "lsq":
        x, w = v["x"].double(), v["w"].double()
        e = x @ w - v["y"].double()
        return {"loss": (e * e).sum(), "dloss/dx": 2.0 * (e @ w.T.contiguous()), "dloss/dw": 2.0 * (x.T.contiguous() @ e)}
    m, t = bs.market, bs.market.maturity
    s0, vol, rate = (float(v[k]) for k in ("s0", "vol", "rate"))
    steps = case.get("steps", 1)
    dt = t / steps
    sums = torch.zeros(3, dtype=torch.float64, device=DEV)
    for z in _normals(case, int(v["seed"])):
        zs = z.sum(1)
        st = s0 * torch.exp((rate - 0.5 * vol * vol) * t + vol * math.sqrt(dt) * zs)
        live = torch.where(st > m.strike, st, torch.zeros_like(st))
        sums += torch.stack([(st - m.strike).clamp_min(0.0).sum(), live.sum() / s0,
                             (live * (math.sqrt(dt) * zs - vol * t)).sum()])
    price, delta, vega = sums * (math.exp(-rate * t) / case["paths"])
    if kind == "price":
        return {"price": price}
    return {"price": price, "dprice/ds0": delta, "dprice/dvol": vega}
