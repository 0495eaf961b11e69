"""The products this library is measured on, through its public entry points.

`listed()` names the cases, `draw(rng)` gives another one of the same ranges,
`prepare` makes what a caller holds before the call (operands on the GPU, a
chain plan), `run` is one call, `work` the bytes and flops the call cannot do
without, `exact` the same result in float64 by plain torch.

Three kinds of case:

* "ttm"   -- one mode-q product, `ttm_amd.ttm`: order 1..5, any layout, extents
             aligned and odd, 1..1024 rows of B, float32 / float64 and the
             float32 precision options;
* "ttms"  -- the multi-TTM of one tensor over every mode but one,
             `ttm_amd.ttmpy.ttms` on device tensors;
* "chain" -- a batch of uneven tensors, each contracted with a factor per mode
             (Tucker cores), one `ChainPlan` replayed as a graph.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

import ttm_amd
from ttm_amd.chain import ChainPlan

DTYPES = {"f32": torch.float32, "f64": torch.float64}
PRECISIONS = ("bf16x3", "fp16x2", "bf16", "fp16", "fp8")


def _ttm(name, na, pi, q, m, dtype="f32", precision="", b="row"):
    return {"name": name, "kind": "ttm", "na": ",".join(map(str, na)), "pi": ",".join(map(str, pi)), "q": q, "m": m,
            "dtype": dtype, "precision": precision, "b": b}


def listed():
    return [
        # the smallest call in use: a 98 304-element tensor, all latency and launches
        _ttm("small-f32", [64, 48, 32], [1, 2, 3], 2, 40, b="col"),
        # compression of one float64 tensor of a few hundred thousand elements
        # over all modes but one: dependent products, each small
        {"name": "ttms-f64", "kind": "ttms", "na": "96,80,112", "q": 2, "r": "24,20,28", "dtype": "f64"},
        # projection of a large tensor to few components, q in the middle of
        # the layout (read-bound)
        _ttm("stream-f32", [1024, 1024, 512], [3, 2, 1], 2, 16),
        # the same along the contiguous mode with odd extents, float64
        _ttm("rows-odd-f64", [515, 641, 766], [1, 2, 3], 1, 10, dtype="f64"),
        # a few dozen components along the contiguous mode
        _ttm("rows-mid-f32", [1024, 1024, 512], [1, 2, 3], 1, 48),
        # order 5 in a permuted layout, every extent short
        _ttm("order5-f32", [32, 24, 40, 16, 48], [4, 2, 3, 1, 5], 3, 64),
        # a large float64 product bound by the matrix cores
        _ttm("large-f64", [1024, 1024, 512], [1, 2, 3], 2, 1024, dtype="f64"),
        # the same size in float32 accuracy on the 16-bit matrix cores
        _ttm("large-bf16x3", [1024, 1024, 512], [1, 2, 3], 2, 1024, precision="bf16x3"),
        # 16-bit operands, contiguous mode, row count between two blocks
        _ttm("large-bf16", [1024, 1024, 512], [3, 2, 1], 3, 800, precision="bf16"),
        # odd extents in the two-term 16-bit precision
        _ttm("odd-fp16x2", [255, 301, 173], [1, 2, 3], 2, 120, precision="fp16x2"),
        # 8-bit operands on an ordinary tensor
        _ttm("mid-fp8", [768, 640, 384], [2, 1, 3], 1, 256, precision="fp8"),
        # Tucker cores of a batch of uneven order-3 tensors
        {"name": "tucker-f32", "kind": "chain", "count": 256, "order": 3, "lo": 16, "hi": 256, "rmax": 64,
         "dtype": "f32", "precision": ""},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extents(rng, p, numel):
    """p extents whose product is near numel; half of them multiples of 16."""
    cuts = [rng.uniform(0.6, 1.4) for _ in range(p)]
    out = []
    for c in cuts:
        n = max(2, int(round(math.exp(math.log(numel) * c / sum(cuts)))))
        if rng.random() < 0.5 and n >= 16:
            n = n // 16 * 16
        out.append(n)
    return out


def draw(rng: random.Random):
    while True:
        kind = rng.choices(["ttm", "low", "ttms", "chain"], [5, 4, 1, 1])[0]
        if kind == "chain":
            dtype, prec = rng.choice([("f32", ""), ("f64", ""), ("f32", "bf16x3"), ("f32", "fp16x2")])
            order = rng.choice([3, 3, 3, 4])
            return {"kind": "chain", "count": _log_int(rng, 8, 256 if dtype == "f32" else 128), "order": order,
                    "lo": 16 if order == 3 else 8, "hi": rng.randint(64, 256) if order == 3 else rng.randint(16, 48),
                    "rmax": rng.randint(8, 64), "dtype": dtype, "precision": prec}
        if kind == "ttms":
            p = rng.choice([3, 4])
            na = _extents(rng, p, _log_int(rng, 1 << 15, 1 << 26))
            r = [max(1, rng.randint(max(1, n // 8), max(1, n // 2))) for n in na]
            return {"kind": "ttms", "na": ",".join(map(str, na)), "q": rng.randint(1, p),
                    "r": ",".join(map(str, r)), "dtype": rng.choice(["f32", "f64"])}
        dtype = rng.choice(["f32", "f32", "f64"]) if kind == "ttm" else "f32"
        prec = "" if kind == "ttm" else rng.choice(PRECISIONS)
        p = rng.choice([1, 2, 3, 3, 3, 4, 5]) if kind == "ttm" else rng.choice([2, 3, 3, 4])
        # p = 1 is a matrix times a vector: B is the large operand there
        na = _extents(rng, p, _log_int(rng, 1 << 14, 1 << 29 if p > 1 else 1 << 22))
        pi = list(range(1, p + 1))
        rng.shuffle(pi)
        q = rng.randint(1, p)
        m = _log_int(rng, 1, 1024) if kind == "ttm" else _log_int(rng, 16, 1024)
        case = _ttm(None, na, pi, q, m, dtype, prec, rng.choice(["row", "col"]))
        del case["name"]
        wk = work(case)
        # within the listed cases' cost and a fifth of the card: in the
        # precision options extents that no 16-byte vector divides stay at
        # ordinary sizes
        w = math.prod(na[r - 1] for r in pi[:pi.index(q)])
        odd = (na[q - 1] if w == 1 else w) % 4 != 0
        if wk["bytes"] <= 9e9 and wk["flops"] <= (4e9 if kind == "low" and odd else 1.1e12):
            return case


# ---------------------------------------------------------------------------
def _ints(text):
    return [int(x) for x in text.split(",")]


def _uniform(gen, shape, dtype):
    """Entries uniform in [-1, 1)."""
    return torch.rand(shape, generator=gen, dtype=dtype, device="cuda").mul_(2).sub_(1)


def _tensor(gen, na, pi, dtype):
    """A dense tensor of extents na in the layout pi (fastest mode first)."""
    slow_first = [r - 1 for r in reversed(pi)]
    store = _uniform(gen, [na[r] for r in slow_first], dtype)
    return store.permute(*[slow_first.index(k) for k in range(len(na))])


def _orthonormal_rows(rng, r, n):
    return np.linalg.qr(rng.standard_normal((n, r)))[0].T


def _operands(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    if case["kind"] == "ttm":
        na, pi = _ints(case["na"]), _ints(case["pi"])
        A = _tensor(gen, na, pi, dtype)
        n = na[case["q"] - 1]
        B = _uniform(gen, (case["m"], n), dtype) if case["b"] == "row" else _uniform(gen, (n, case["m"]), dtype).t()
        return A, B
    nprng = np.random.default_rng(seed)

    def factor(r, n):
        return torch.from_numpy(np.ascontiguousarray(_orthonormal_rows(nprng, r, n))).to("cuda", dtype)

    if case["kind"] == "ttms":
        na, r = _ints(case["na"]), _ints(case["r"])
        A = _uniform(gen, na, dtype)
        return A, [factor(r[k], na[k]) for k in range(len(na)) if k != case["q"] - 1]
    # the extents and ranks are the case's, the same for every seed
    shapes = random.Random(case["count"] * 1000 + case["hi"])
    tensors, factors = [], []
    for _ in range(case["count"]):
        na = [shapes.randint(case["lo"], case["hi"]) for _ in range(case["order"])]
        r = [min(n, shapes.randint(4, case["rmax"])) for n in na]
        tensors.append(_tensor(gen, na, list(range(1, len(na) + 1)), dtype))
        factors.append([factor(rk, n) for rk, n in zip(r, na)])
    return tensors, factors


def _padded(extents):
    return -(-math.prod(extents) // 64) * 64


def prepare(case, seed):
    X, Y = _operands(case, seed)
    state = {"case": case, "A": X, "B": Y}
    if case["kind"] == "chain":
        # the cores of the batch in one buffer, each at a 256-byte boundary
        ranks = [[U.shape[0] for U in Us] for Us in Y]
        pad = [_padded(rk) for rk in ranks]
        state["C"] = torch.zeros(sum(pad), dtype=X[0].dtype, device="cuda")
        items, at = [], 0
        for A, Us, rk, n in zip(X, Y, ranks, pad):
            pi = ttm_amd.layout_from_strides(list(A.shape), list(A.stride()))
            items.append((A, Us, torch.as_strided(state["C"], rk, ttm_amd.dense_strides(rk, pi), at)))
            at += n
        state["plan"] = ChainPlan(items, precision=case["precision"] or None)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "ttm":
        return ttm_amd.ttm(case["q"], state["A"], state["B"], b_layout=case["b"], precision=case["precision"] or None)
    if case["kind"] == "ttms":
        return ttm_amd.ttmpy.ttms(case["q"], state["A"], state["B"], "forward")
    state["plan"].run_graph()
    return state["C"]


def _chain_work(na, r, modes, size):
    flops, nb = 0, 0
    cur = list(na)
    for k in modes:
        flops += 2 * r[k] * math.prod(cur)
        nb += r[k] * cur[k]
        cur[k] = r[k]
    return size * (math.prod(na) + nb + math.prod(cur)), flops


def work(case):
    size = 8 if case["dtype"] == "f64" else 4
    if case["kind"] == "ttm":
        na, m = _ints(case["na"]), case["m"]
        numel, n = math.prod(na), na[case["q"] - 1]
        return {"bytes": size * (numel + m * n + numel // n * m), "flops": 2 * m * numel}
    if case["kind"] == "ttms":
        na, r = _ints(case["na"]), _ints(case["r"])
        b, f = _chain_work(na, r, [k for k in range(len(na)) if k != case["q"] - 1], size)
        return {"bytes": b, "flops": f}
    shapes = random.Random(case["count"] * 1000 + case["hi"])
    total_b = total_f = 0
    for _ in range(case["count"]):
        na = [shapes.randint(case["lo"], case["hi"]) for _ in range(case["order"])]
        r = [min(n, shapes.randint(4, case["rmax"])) for n in na]
        b, f = _chain_work(na, r, range(len(na)), size)
        total_b, total_f = total_b + b, total_f + f
    return {"bytes": total_b, "flops": total_f}


def _product64(A, B, q):
    """A x_q B in float64: modes other than q as rows of one matrix product."""
    X = A.movedim(q - 1, -1)
    Y = X.reshape(-1, X.shape[-1]).to(torch.float64) @ B.to(torch.float64).t().contiguous()
    return Y.reshape(*X.shape[:-1], B.shape[0]).movedim(-1, q - 1)


def exact(case, seed):
    X, Y = _operands(case, seed)
    if case["kind"] == "ttm":
        return _product64(X, Y, case["q"])
    if case["kind"] == "ttms":
        modes = [k for k in range(1, X.dim() + 1) if k != case["q"]]
        for k, U in zip(modes, Y):
            X = _product64(X, U, k)
        return X
    pad = [_padded([U.shape[0] for U in Us]) for Us in Y]
    out = torch.zeros(sum(pad), dtype=torch.float64, device="cuda")
    at = 0
    for A, Us, n in zip(X, Y, pad):
        for k, U in enumerate(Us):
            A = _product64(A, U, k + 1)
        # first-order layout: mode 1 fastest
        flat = A.permute(*reversed(range(A.dim()))).reshape(-1)
        out[at:at + flat.numel()] = flat
        at += n
    return out
