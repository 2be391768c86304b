"""The array programs whose speed is measured: what each stands for, its inputs, one pass, and its values in 64 bits.

Every case is a program against the public front end (`bohrium_amd`): the benchmark programs of
`bohrium_amd.workloads` and the building blocks that its random programs are made of.  Kinds:

    small      a map and a sum over an array of a few thousand elements: what one short program costs (launches, flush)
    stream     one fused block over a large array: the map x*2+1, its sum, or max|x-0.5|
    mc_pi      Monte-Carlo pi: two philox draws per point, an int64 count
    pricing    fused Black-Scholes pricing in float64, one sum per time step, the steps one do_while
    heat       the 5-point Jacobi stencil in place with max|new-old| per sweep, the sweeps one do_while or a loop of
               flushes
    rows       mean and variance of every row (axis 1) and the standardised matrix
    columns    the same of every column (axis 0): a table of samples by features
    scan       running count of x > 0 (int64) or running sum (float64) of a vector
    views      element-wise work on transposed, reversed and half views of one matrix
    matmul     matrix products of the four BLAS types
    batched    many short arrays of uneven sizes in one flush: map, sum, running count, gather

Inputs are made by torch on the GPU from the seed and copied into arrays of the engine; results stay in
device memory and are looked at through the pointer that the engine hands out, except scalars, which a
program fetches.
"""
import math

import numpy as np
import torch

import bohrium_amd as bh
from bohrium_amd import _bh_api, workloads

_DTYPES = {"float32": (np.float32, torch.float32), "float64": (np.float64, torch.float64),
           "complex64": (np.complex64, torch.complex64), "complex128": (np.complex128, torch.complex128)}
_BYTES = {"float32": 4, "float64": 8, "complex64": 8, "complex128": 16}
_BLACK_SCHOLES = {"r": 0.02, "sigma": 0.3, "dt": 0.01}
_EPS = 1e-5  # added to the variances of `rows` and `columns`


def listed():
    return [
        # A short program on a short vector: flush, launches and the fetch of one number count, not bandwidth.
        {"name": "small_vector", "kind": "small", "n": 1000, "dtype": "float64"},
        # The memory-bound fused block of the streaming benchmark (1 GiB read, 1 GiB written).
        {"name": "stream_map", "kind": "stream", "op": "map", "n": 1 << 28, "dtype": "float32"},
        # Monte-Carlo pi of the benchmark: 1e7 points, integer arithmetic.
        {"name": "mc_pi", "kind": "mc_pi", "n": 10_000_000},
        # The headline benchmark: option pricing of 2e7 contracts, 10 time steps.
        {"name": "pricing", "kind": "pricing", "n": 20_000_000, "steps": 10},
        # The heat stencil of the benchmark: 8192 x 8192, 200 sweeps (the largest case).
        {"name": "heat", "kind": "heat", "rows": 8192, "cols": 8192, "sweeps": 200, "dtype": "float32",
         "loop": "do_while"},
        # Row statistics of a matrix (axis 1), as in the random programs, at a row length that is no power of two.
        {"name": "rows", "kind": "rows", "rows": 16384, "cols": 3000, "dtype": "float32"},
        # Column statistics (axis 0) of a tall table of samples by features.
        {"name": "columns", "kind": "columns", "rows": 100_000, "cols": 500, "dtype": "float32"},
        # Running count over a long vector of odd length.
        {"name": "scan_count", "kind": "scan", "op": "count", "n": 60_000_001},
        # Transposed, reversed and half views of a square matrix, as in the random programs.
        {"name": "views", "kind": "views", "side": 4096, "dtype": "float32"},
        # A square matrix product in float64.
        {"name": "matmul_f64", "kind": "matmul", "m": 4096, "n": 4096, "k": 4096, "dtype": "float64"},
        # A rectangular complex product with ragged edges.
        {"name": "matmul_c128", "kind": "matmul", "m": 2000, "n": 1500, "k": 2500, "dtype": "complex128"},
        # Uneven short arrays in one flush (the batched benchmark's programs and sizes).
        {"name": "batched", "kind": "batched", "count": 20, "lo": 256, "hi": 262144},
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, spread evenly over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["small", "stream", "mc_pi", "pricing", "heat", "rows", "columns", "scan", "views", "matmul",
                       "batched"])
    real = rng.choice(["float32", "float64"])
    if kind == "small":
        return {"kind": kind, "n": _spread(rng, 2, 65536), "dtype": real}
    if kind == "stream":
        return {"kind": kind, "op": rng.choice(["map", "sum", "maxabs"]), "dtype": real,
                "n": _spread(rng, 65536, 1 << 28 if real == "float32" else 1 << 27)}
    if kind == "mc_pi":
        return {"kind": kind, "n": _spread(rng, 10_000, 10_000_000)}
    if kind == "pricing":
        return {"kind": kind, "n": _spread(rng, 10_000, 20_000_000), "steps": rng.randint(2, 10)}
    if kind == "heat":
        rows, cols = _spread(rng, 128, 8192), _spread(rng, 128, 8192)
        return {"kind": kind, "rows": rows, "cols": cols, "dtype": real, "sweeps": rng.randint(10, 100), "loop": "flushes"}
    if kind in ("rows", "columns"):
        along = _spread(rng, 16, 200_000)
        across = _spread(rng, 8, max(8, min(65536, (1 << 26) // along)))
        rows, cols = (across, along) if kind == "rows" else (along, across)
        return {"kind": kind, "rows": rows, "cols": cols, "dtype": real}
    if kind == "scan":
        return {"kind": kind, "op": rng.choice(["count", "sum"]), "n": _spread(rng, 1000, 1 << 26)}
    if kind == "views":
        return {"kind": kind, "side": _spread(rng, 64, 4096), "dtype": real}
    if kind == "matmul":
        return {"kind": kind, "m": _spread(rng, 16, 4096), "n": _spread(rng, 16, 4096), "k": _spread(rng, 16, 4096),
                "dtype": rng.choice(sorted(_DTYPES))}
    return {"kind": "batched", "count": rng.randint(9, 21), "lo": 256, "hi": _spread(rng, 1024, 262144)}


# ---------------------------------------------------------------- inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, shape, dtype):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _between(g, lo, hi, shape, dtype=torch.float64):
    return torch.rand(shape, generator=g, device="cuda", dtype=dtype) * (hi - lo) + lo


def _drawn(case, seed):
    """The inputs of a case as torch tensors, by name."""
    g, kind = _generator(seed), case["kind"]
    t = _DTYPES[case["dtype"]][1] if "dtype" in case else None
    if kind == "mc_pi":
        return {}
    if kind in ("small", "stream"):
        return {"x": torch.rand(case["n"], generator=g, device="cuda", dtype=t)}
    if kind == "pricing":
        n = case["n"]
        return {"S": _between(g, 58.0, 62.0, n), "K": _between(g, 55.0, 65.0, n), "T": _between(g, 0.25, 2.0, n)}
    if kind == "heat":
        grid = _between(g, -20.0, 20.0, (case["rows"], case["cols"]), t)
        grid[:, 0] = grid[:, -1] = -273.0
        grid[-1, :] = -273.0
        grid[0, :] = 40.0
        return {"grid": grid, "delta": torch.zeros((1,), device="cuda", dtype=t)}
    if kind in ("rows", "columns"):
        return {"x": _normal(g, (case["rows"], case["cols"]), t) * 2.0 + 1.0}
    if kind == "scan":
        return {"x": _normal(g, case["n"], torch.float32 if case["op"] == "count" else torch.float64)}
    if kind == "views":
        return {"a": _normal(g, (case["side"], case["side"]), t)}
    if kind == "matmul":
        return {"a": _normal(g, (case["m"], case["k"]), t), "b": _normal(g, (case["k"], case["n"]), t)}
    out = {}
    for i, n in enumerate(_sizes(case)):
        out["x%d" % i] = _normal(g, n, torch.float32)
        out["i%d" % i] = torch.randint(0, n, (n,), generator=g, device="cuda", dtype=torch.int64)
    return out


def _sizes(case):
    return [int(n) for n in workloads.batched_sizes(case["count"], case["lo"], case["hi"])]


class _Memory:
    """A contiguous array's device memory for torch (it keeps the array alive)."""

    def __init__(self, array):
        self.array = array
        self.__cuda_array_interface__ = {"shape": array.shape, "typestr": array.dtype.str, "strides": None, "version": 3,
                                         "data": (_bh_api.data_get(array.base.handle, copy2host=False), False)}


def _tensor(array):
    return torch.as_tensor(_Memory(array), device="cuda")


def _arrays(tensors):
    """Arrays of the engine with the values of `tensors`, in device memory."""
    out = {}
    for name, t in tensors.items():
        out[name] = bh.zeros(tuple(t.shape), np.dtype(str(t.dtype).replace("torch.", "")))
    bh.flush()
    torch.cuda.synchronize()
    for name, t in tensors.items():
        _tensor(out[name]).copy_(t)
    torch.cuda.synchronize()
    return out


_SETTLED = set()


def _trials():
    for line in bh.message("statistic").splitlines():
        if line.startswith("autotune_trials:"):
            return float(line.split(":")[1])
    return 0.0


def _settle(case, seed):
    """Runs the program on inputs of its own until the engine's autotuner tries no more launch shapes: the
    plan that a long-running program keeps."""
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key in _SETTLED:
        return
    state = {"case": case, "seed": seed, **_arrays(_drawn(case, seed))}
    for _ in range(100):
        before = _trials()
        run(state)
        torch.cuda.synchronize()
        if _trials() == before:
            break
    bh.message("autotune")
    run(state)
    torch.cuda.synchronize()
    _SETTLED.add(key)


def prepare(case, seed):
    _settle(case, seed)
    return {"case": case, "seed": seed, **_arrays(_drawn(case, seed))}


# ---------------------------------------------------------------- one pass

def _standardise(x, axis):
    m = x.mean(axis)
    c = x - (m[None, :] if axis == 0 else m[:, None])
    v = (c * c).mean(axis)
    s = bh.sqrt(v + _EPS)
    z = c / (s[None, :] if axis == 0 else s[:, None])
    return z, m, v


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "small":
        y = state["x"] * 2 + 1
        total = y.sum().asnumpy()
        return _tensor(y), total
    if kind == "stream":
        x = state["x"]
        if case["op"] == "map":
            z = x * 2 + 1
            bh.flush()
            return _tensor(z)
        return ((x * 2 + 1).sum() if case["op"] == "sum" else bh.abs(x - 0.5).max()).asnumpy()
    if kind == "mc_pi":
        return workloads.mc_pi(case["n"], state["seed"]).asnumpy()
    if kind == "pricing":
        return _tensor(workloads.black_scholes_repeat(state["S"], state["K"], state["T"], case["steps"], **_BLACK_SCHOLES))
    if kind == "heat":
        grid, delta = state["grid"], state["delta"]

        def sweep():
            delta[...] = workloads.jacobi_step(grid)

        if case["loop"] == "do_while":
            bh.do_while(sweep, case["sweeps"])
        else:
            for _ in range(case["sweeps"]):
                sweep()
                bh.flush()
        return _tensor(grid), _tensor(delta)
    if kind in ("rows", "columns"):
        out = _standardise(state["x"], 1 if kind == "rows" else 0)
        bh.flush()
        return [_tensor(a) for a in out]
    if kind == "scan":
        x = state["x"]
        y = (x > 0).astype(np.int64).cumsum() if case["op"] == "count" else x.cumsum()
        bh.flush()
        return _tensor(y)
    if kind == "views":
        a = state["a"]
        h = a.shape[0] // 2
        out = [(a + a.T) * 0.5, a[::-1, :] - a[:, ::-1], a[:h] + a[h:2 * h], a.T * 1.0]
        bh.flush()
        return [_tensor(v) for v in out]
    if kind == "matmul":
        c = bh.matmul(state["a"], state["b"])
        bh.flush()
        return _tensor(c)
    n = case["count"]
    out = workloads.batched_step([state["x%d" % i] for i in range(n)], [state["i%d" % i] for i in range(n)])
    sums = bh.asnumpy_many(out[0])
    return {"sums": np.array(sums), "counts": [_tensor(c) for c in out[1]], "gathered": [_tensor(y) for y in out[2]]}


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    kind = case["kind"]
    b = _BYTES.get(case.get("dtype"), 0)
    if kind == "small" or (kind == "stream" and case["op"] == "map"):
        return {"bytes": 2 * b * case["n"], "flops": 2 * case["n"]}
    if kind == "stream":
        return {"bytes": b * case["n"], "flops": 3 * case["n"]}
    if kind == "mc_pi":
        # two counter-based draws of ten rounds (about 4 operations each) and the test
        return {"bytes": 8, "flops": 84 * case["n"]}
    if kind == "pricing":
        # about 70 array operations per contract and step, exp, log and sqrt counted as one each
        return {"bytes": 24 * case["n"] * case["steps"], "flops": 70 * case["n"] * case["steps"]}
    if kind == "heat":
        r, c = case["rows"], case["cols"]
        return {"bytes": case["sweeps"] * b * (r * c + (r - 2) * (c - 2)), "flops": 8 * case["sweeps"] * (r - 2) * (c - 2)}
    if kind in ("rows", "columns"):
        r, c = case["rows"], case["cols"]
        return {"bytes": b * (2 * r * c + 2 * (r if kind == "rows" else c)), "flops": 6 * r * c}
    if kind == "scan":
        return {"bytes": (12 if case["op"] == "count" else 16) * case["n"], "flops": case["n"]}
    if kind == "views":
        s = case["side"]
        return {"bytes": b * (4 * s * s + (s // 2) * s), "flops": 5 * s * s}
    if kind == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": b * (m * k + k * n + m * n), "flops": (8 if case["dtype"].startswith("complex") else 2) * m * n * k}
    elems = sum(_sizes(case))
    return {"bytes": 24 * elems, "flops": 6 * elems}


def tolerance(case):
    """About four times the differences that were measured: from the values in 64 bits, or where the two largest of
    the range were not at hand, what the type's sums give over the range's lengths."""
    kind, dtype = case["kind"], case.get("dtype")
    single = dtype in ("float32", "complex64")
    if kind == "mc_pi" or (kind == "scan" and case["op"] == "count"):
        return "exact"
    if kind == "pricing":
        return {"rel": 1e-13}
    if kind == "scan":
        return {"rel": 1e-13}  # order of the sums (tiles look back as far as they find a prefix)
    if kind == "heat":
        # max|new - old| is a difference of numbers up to two thousand times its size
        return {"rel": 5e-4 if single else 1e-12}
    if kind == "stream" and case["op"] == "sum":
        return {"rel": 1e-5 if single else 1e-13}
    if kind == "matmul":
        return {"rel": 4e-6 if single else 1e-14}
    if kind == "batched":
        return {"rel": 1e-6}
    return {"rel": 1e-6 if single else 1e-14}


# ---------------------------------------------------------------- the same in 64 bits

def _cnd(d):
    k = 1.0 / (d.abs() * workloads.CND_P + 1.0)
    a1, a2, a3, a4, a5 = workloads.CND_A
    poly = k * (a1 + k * (a2 + k * (a3 + k * (a4 + k * a5))))
    w = 1.0 - workloads.RSQRT2PI * torch.exp(d * d * -0.5) * poly
    return torch.where(d < 0.0, 1.0 - w, w)


def exact(case, seed):
    kind = case["kind"]
    if kind == "mc_pi":
        return None
    t = {k: v.to(torch.complex128 if v.is_complex() else torch.float64) if not k.startswith("i") else v
         for k, v in _drawn(case, seed).items()}
    if kind == "small":
        y = t["x"] * 2 + 1
        return y, y.sum().cpu().numpy()
    if kind == "stream":
        x = t["x"]
        if case["op"] == "map":
            return x * 2 + 1
        return ((x * 2 + 1).sum() if case["op"] == "sum" else (x - 0.5).abs().max()).cpu().numpy()
    if kind == "pricing":
        S, K, T = t["S"], t["K"], t["T"]
        r, sigma, dt = (_BLACK_SCHOLES[k] for k in ("r", "sigma", "dt"))
        sums = []
        for i in range(case["steps"]):
            Tt = T + i * dt
            sq = torch.sqrt(Tt)
            d1 = (torch.log(S / K) + (r + 0.5 * sigma * sigma) * Tt) / (sigma * sq)
            sums.append((S * _cnd(d1) - K * torch.exp(Tt * -r) * _cnd(d1 - sigma * sq)).sum())
        return torch.stack(sums)
    if kind == "heat":
        G = t["grid"]
        for _ in range(case["sweeps"]):
            new = (G[1:-1, 1:-1] + G[:-2, 1:-1] + G[2:, 1:-1] + G[1:-1, :-2] + G[1:-1, 2:]) * 0.2
            delta = (new - G[1:-1, 1:-1]).abs().max()
            G[1:-1, 1:-1] = new
        return G, delta.reshape(1)
    if kind in ("rows", "columns"):
        x, axis = t["x"], 1 if kind == "rows" else 0
        m = x.mean(axis, keepdim=True)
        c = x - m
        v = (c * c).mean(axis, keepdim=True)
        return [c / torch.sqrt(v + _EPS), m.squeeze(axis), v.squeeze(axis)]
    if kind == "scan":
        return None if case["op"] == "count" else torch.cumsum(t["x"], 0)
    if kind == "views":
        a = t["a"]
        h = a.shape[0] // 2
        return [(a + a.T) * 0.5, a.flip(0) - a.flip(1), a[:h] + a[h:2 * h], a.T.contiguous()]
    if kind == "matmul":
        return t["a"] @ t["b"]
    sums, gathered = [], []
    for i in range(case["count"]):
        y = torch.tanh(t["x%d" % i] * 0.5 + 0.1)
        sums.append(float(y.sum()))
        gathered.append(y[t["i%d" % i]])
    return {"sums": np.array(sums), "counts": [None] * case["count"], "gathered": gathered}
