"""The work whose speed counts: products of sparse matrices as programs call them.

Each case is a dict of plain values naming a kind of work and its sizes:

  layer    C = A B, A a pruned weight matrix, B the activations (one column per
           token): planned once, run per batch.  Rows alike ("uniform") or of
           very different lengths ("lognormal").
  graph    C = A B, A the normalised adjacency of a power-law graph (R-MAT,
           symmetric, self-loops), B node features: planned once on the GPU.
  zipf     C = A B with a few very long rows and most rows empty.
  train_graph, train_layer
           forward and backward of the differentiable operator: C, the
           gradient of A's values and the gradient of B.
  bell     C = A B, A block-sparse in Blocked-ELL.
  s24      C = A B, A compressed 2:4.
  sampled  a sampled neighbourhood: a new structure on the GPU each pass,
           planned there and multiplied once.

Inputs come from the seed alone and are made on the GPU with torch.
"""
import math

import numpy as np
import torch

import spmm_amd as S
from spmm_amd import torch_ops as T

DEV = "cuda:0"
TORCH = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
TCA = {"f16": S.TCA_F16, "bf16": S.TCA_BF16, "f32": S.TCA_F32}
SIZE = {"f16": 2, "bf16": 2, "f32": 4}
RMAT = (0.57, 0.19, 0.19)  # quadrant probabilities of the graphs, the fourth is the rest


def listed():
    return [
        # smallest: a 90 % pruned feed-forward matrix with a short inner size; one launch of a few microseconds
        {"name": "layer_small", "kind": "layer", "m": 2048, "k": 512, "density": 0.1, "rows": "uniform", "n": 256,
         "dtype": "f16"},
        # prefill of a pruned square layer whose rows keep very different shares
        {"name": "layer_prefill", "kind": "layer", "m": 4096, "k": 4096, "density": 0.05, "rows": "lognormal",
         "n": 512, "dtype": "f16"},
        # decode: the same kind of layer, one token
        {"name": "layer_decode", "kind": "layer", "m": 8192, "k": 8192, "density": 0.1, "rows": "uniform", "n": 1,
         "dtype": "f16"},
        # a batch of an odd number of tokens through a layer of odd sizes
        {"name": "layer_ragged", "kind": "layer", "m": 3001, "k": 2049, "density": 0.08, "rows": "uniform", "n": 333,
         "dtype": "bf16"},
        # aggregation of a social graph (233k nodes, 115M edges) at a hidden width of 128
        {"name": "graph_hidden", "kind": "graph", "nodes": 232965, "edges": 90800000, "n": 128, "dtype": "f32"},
        # the last layer of a product graph (2.4M nodes, 64M edges): as many columns as there are classes
        {"name": "graph_classes", "kind": "graph", "nodes": 2449029, "edges": 32150000, "n": 47, "dtype": "f32"},
        # a million rows, 20M entries, most of them in a few hundred rows
        {"name": "zipf", "kind": "zipf", "m": 1 << 20, "k": 1 << 20, "total": 20000000, "n": 64, "dtype": "f16"},
        # a training step over a graph whose edge weights are learned
        {"name": "train_graph", "kind": "train_graph", "nodes": 131072, "edges": 8000000, "n": 128, "dtype": "f32"},
        # a training step of a sparse layer: forward, weight gradient, input gradient
        {"name": "train_layer", "kind": "train_layer", "m": 2048, "k": 2048, "density": 0.1, "rows": "uniform",
         "n": 1024, "dtype": "bf16"},
        # block-sparse layer, a quarter of its 32 x 32 blocks kept
        {"name": "bell", "kind": "bell", "m": 4096, "k": 4096, "block": 32, "density": 0.25, "n": 512,
         "dtype": "f16"},
        # 2:4 pruned layer
        {"name": "s24", "kind": "s24", "m": 4096, "k": 4096, "n": 512, "dtype": "bf16"},
        # minibatch of a sampled neighbourhood: plan on the GPU, multiply once
        {"name": "sampled", "kind": "sampled", "m": 20000, "k": 100000, "fanout": 15, "n": 128, "dtype": "f32"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A width: powers of two, multiples of 8 and odd ones alike."""
    n = _log(rng, lo, hi)
    pick = rng.random()
    if pick < 0.35:
        return 1 << max(0, round(math.log2(n)))
    if pick < 0.6 and n >= 8:
        return n // 8 * 8
    return n


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "graph", "graph", "zipf", "train_graph", "train_layer", "bell",
                       "s24", "sampled"])
    half = rng.choice(["f16", "bf16"])
    any_type = rng.choice(["f32", "f32", "f16", "bf16"])
    if kind in ("layer", "train_layer"):
        top = 12000 if kind == "layer" else 4096
        case = {"kind": kind, "m": _log(rng, 300, top), "k": _log(rng, 200, top),
                "density": round(math.exp(rng.uniform(math.log(0.02), math.log(0.3))), 3),
                "rows": rng.choice(["uniform", "lognormal"]),
                "n": _width(rng, 1 if kind == "layer" else 16, 1024), "dtype": rng.choice([half, half, any_type])}
        while case["m"] * case["k"] * case["density"] * case["n"] > 4e9:
            case["n"] = (case["n"] + 1) // 2
        return case
    if kind in ("graph", "train_graph"):
        nodes = _log(rng, 3000, 1500000 if kind == "graph" else 200000)
        edges = int(nodes * _log(rng, 3, 100 if kind == "graph" else 60))
        case = {"kind": kind, "nodes": nodes, "edges": min(edges, 20000000 if kind == "graph" else 8000000),
                "n": _width(rng, 7, 256 if kind == "graph" else 128), "dtype": any_type}
        while case["edges"] * case["n"] > 1.5e9:
            case["n"] = (case["n"] + 1) // 2
        return case
    if kind == "zipf":
        m = _log(rng, 20000, 1 << 20)
        return {"kind": kind, "m": m, "k": _log(rng, 20000, 1 << 20), "total": min(m * rng.randint(2, 20), 20000000),
                "n": _width(rng, 8, 128), "dtype": any_type}
    if kind == "bell":
        return {"kind": kind, "m": _log(rng, 256, 6000), "k": _log(rng, 256, 6000), "block": rng.choice([32, 64]),
                "density": round(rng.uniform(0.05, 0.5), 3), "n": 8 * _log(rng, 1, 128), "dtype": half}
    if kind == "s24":
        return {"kind": kind, "m": _log(rng, 256, 6000), "k": _log(rng, 256, 6000), "n": 8 * _log(rng, 1, 128),
                "dtype": half}
    m = _log(rng, 1000, 60000)
    return {"kind": "sampled", "m": m, "k": m * rng.randint(2, 8), "fanout": rng.randint(5, 25),
            "n": _width(rng, 16, 256), "dtype": any_type}


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 1000003 + 17)
    return g


def _csr_from_keys(keys, m, k):
    """Row offsets and columns (int32) of the sorted entry keys row * k + col."""
    rows = torch.div(keys, k, rounding_mode="floor")
    rowptr = torch.zeros(m + 1, dtype=torch.int64, device=DEV)
    rowptr[1:] = torch.cumsum(torch.bincount(rows, minlength=m), 0)
    return rowptr.to(torch.int32), (keys - rows * k).to(torch.int32)


def _layer_pattern(case, g):
    m, k = case["m"], case["k"]
    score = torch.rand((m, k), generator=g, device=DEV)
    if case["rows"] == "lognormal":  # a row's entries come first by a factor of its own
        score /= torch.exp(torch.randn((m, 1), generator=g, device=DEV))
    keep = torch.sort(score.flatten()).indices[:int(_entries(case))]
    return _csr_from_keys(torch.sort(keep).values, m, k)


def _levels(nodes):
    return max(1, math.ceil(math.log2(nodes)))


def _graph_pattern(case, g):
    n, s = case["nodes"], case["edges"]
    a, b, c = RMAT
    kept, have = [torch.arange(n, device=DEV) * (n + 1)], 0  # the loops, then the sampled edges both ways
    while have < s:
        u = torch.zeros(s, dtype=torch.int64, device=DEV)
        v = torch.zeros(s, dtype=torch.int64, device=DEV)
        for _ in range(_levels(n)):
            r = torch.rand(s, generator=g, device=DEV)
            u = u * 2 + (r >= a + b)
            v = v * 2 + (((r >= a) & (r < a + b)) | (r >= a + b + c))
        ok = (u < n) & (v < n) & (u != v)
        u, v = u[ok][:s - have], v[ok][:s - have]
        kept += [u * n + v, v * n + u]
        have += u.numel()
    keys = torch.unique(torch.cat(kept))
    if case["kind"] == "train_graph":  # as many for every seed: some are left out again
        keep = torch.sort(torch.randperm(keys.numel(), generator=g, device=DEV)[:int(_entries(case))]).values
        keys = keys[keep]
    return _csr_from_keys(keys, n, n)


def _zipf_pattern(case, g):
    m, k, total = case["m"], case["k"], case["total"]
    u = torch.rand(m, generator=g, device=DEV, dtype=torch.float64).clamp_min(1e-12)
    raw = torch.floor(u ** -2.0)  # Zipf of exponent 1.5
    cap = float(min(200000, k // 4))
    lo, hi = 0.0, 1.0
    for _ in range(50):  # the largest factor that keeps the total
        f = (lo + hi) / 2
        if float(torch.clamp(torch.floor(raw * f), max=cap).sum()) > total:
            hi = f
        else:
            lo = f
    length = torch.clamp(torch.floor(raw * lo), max=cap).to(torch.int64)
    rows = torch.repeat_interleave(torch.arange(m, device=DEV), length)
    cols = torch.randint(0, k, (rows.numel(),), generator=g, device=DEV)
    return _csr_from_keys(torch.unique(rows * k + cols), m, k)


def _sampled_pattern(case, g):
    m, k, f = case["m"], case["k"], case["fanout"]
    cols = torch.randint(0, k, (m, f), generator=g, device=DEV)
    some = torch.rand((m, f), generator=g, device=DEV) < 0.9  # some nodes have fewer neighbours
    rows = torch.arange(m, device=DEV)[:, None]
    return _csr_from_keys(torch.unique((rows * k + cols)[some]), m, k)


def _rows_of(rowptr):
    lens = (rowptr[1:] - rowptr[:-1]).to(torch.int64)
    return torch.repeat_interleave(torch.arange(lens.numel(), device=DEV), lens)


def _shape(case):
    return (case["nodes"], case["nodes"]) if "nodes" in case else (case["m"], case["k"])


def _inputs(case, seed):
    """(rowptr, colidx, values, B, G): A as a CSR on the GPU, the dense operand
    and, for training, the gradient of C that arrives from above."""
    g = _generator(seed)
    kind, dt = case["kind"], TORCH[case["dtype"]]
    m, k = _shape(case)
    pattern = {"layer": _layer_pattern, "train_layer": _layer_pattern, "graph": _graph_pattern,
               "train_graph": _graph_pattern, "zipf": _zipf_pattern, "sampled": _sampled_pattern}[kind]
    rowptr, colidx = pattern(case, g)
    nnz = colidx.numel()
    deg = (rowptr[1:] - rowptr[:-1]).clamp_min(1).to(torch.float32)
    if kind in ("graph", "train_graph"):  # D^-1/2 A D^-1/2
        values = (deg.rsqrt()[_rows_of(rowptr)] * deg.rsqrt()[colidx.long()]).to(dt)
    elif kind == "sampled":  # mean over the sampled neighbours
        values = (1.0 / deg)[_rows_of(rowptr)].to(dt)
    elif kind == "zipf":
        values = (torch.rand(nnz, generator=g, device=DEV) * 2 - 1).to(dt)
    else:
        values = (torch.randn(nnz, generator=g, device=DEV) * 0.02).to(dt)
    b = torch.randn((k, case["n"]), generator=g, device=DEV).to(dt)
    gc = torch.randn((m, case["n"]), generator=g, device=DEV) if kind.startswith("train") else None
    return rowptr, colidx, values, b, gc


def _dense_inputs(case, seed):
    """(dense A, B) of the block and 2:4 cases, A's zeros explicit."""
    g = _generator(seed)
    m, k, dt = case["m"], case["k"], TORCH[case["dtype"]]
    a = torch.randn((m, k), generator=g, device=DEV) * 0.02
    if case["kind"] == "bell":
        bs = case["block"]
        rows, cols = -(-m // bs), -(-k // bs)
        keep = torch.rand((rows, cols), generator=g, device=DEV) < case["density"]
        a = a * keep.repeat_interleave(bs, 0)[:m].repeat_interleave(bs, 1)[:, :k]
    else:  # the two largest of every four columns
        kp = -(-k // 4) * 4
        q = torch.zeros((m, kp), device=DEV)
        q[:, :k] = a.abs()
        top = torch.zeros((m, kp // 4, 4), dtype=torch.bool, device=DEV)
        top.scatter_(2, q.view(m, kp // 4, 4).topk(2, 2).indices, True)
        a = a * top.view(m, kp)[:, :k]
    b = torch.randn((k, case["n"]), generator=g, device=DEV).to(dt)
    return a.to(dt), b


def _host(t):
    """A tensor as the numpy storage of the package (16-bit patterns for bf16)."""
    t = t.cpu()
    return t.view(torch.int16).numpy().view(np.uint16) if t.dtype == torch.bfloat16 else t.numpy()


def _device(x, dtype):
    x = np.ascontiguousarray(x)
    return torch.from_numpy(x.view(np.int16)).to(DEV).view(TORCH[dtype])


def _host_csr(case, rowptr, colidx, values):
    m, k = _shape(case)
    return S.CSR(m, k, _host(rowptr), _host(colidx), _host(values), TCA[case["dtype"]])


# ------------------------------------------------------------------ a program's calls
def prepare(case, seed):
    kind, n, dt = case["kind"], case["n"], case["dtype"]
    m, k = _shape(case)
    c = torch.empty((m, n), dtype=torch.float32, device=DEV)
    if kind in ("bell", "s24"):
        a, b = _dense_inputs(case, seed)
        keys = a.flatten().nonzero().flatten()
        csr = _host_csr(case, *_csr_from_keys(keys, m, k), a.flatten()[keys])
        if kind == "bell":
            colind, vals = S.csr_to_bell(csr, case["block"])
            return {"case": case, "colind": torch.from_numpy(colind).to(DEV), "values": _device(vals, dt), "b": b,
                    "c": c}
        vals, meta = S.csr_to_24(csr)
        return {"case": case, "values": _device(vals, dt), "meta": torch.from_numpy(meta.view(np.int16)).to(DEV),
                "b": b, "c": c}
    rowptr, colidx, values, b, gc = _inputs(case, seed)
    state = {"case": case, "values": values, "b": b, "c": c}
    if kind == "sampled":
        state.update(rowptr=rowptr, colidx=colidx)
    elif kind == "graph":
        state["plan"] = S.Plan.from_device(rowptr, colidx, m, k, colidx.numel(), n, TCA[dt])
    elif kind in ("layer", "zipf"):
        state["plan"] = S.Plan(_host_csr(case, rowptr, colidx, values), n)
    else:
        sm = T.SparseMatrix(_host_csr(case, rowptr, colidx, values), DEV)
        sm.plan(n), sm.plan_t(n)  # a training program's first step plans both directions
        state.update(matrix=sm, values=values.requires_grad_(), b=b.requires_grad_(), gc=gc)
    return state


def run(state):
    case = state["case"]
    kind, n, dt = case["kind"], case["n"], TCA[case["dtype"]]
    if kind.startswith("train"):
        c = T.spmm(state["matrix"], state["values"], state["b"])
        gv, gb = torch.autograd.grad(c, (state["values"], state["b"]), state["gc"])
        return {"c": c.detach(), "grad_values": gv, "grad_b": gb}
    stream = torch.cuda.current_stream().cuda_stream
    m, k = _shape(case)
    c = state["c"]
    if kind == "bell":
        S.bell_spmm(state["colind"], state["values"], m, k, n, case["block"], dt, state["b"], c, stream=stream)
    elif kind == "s24":
        S.spmm_24(state["values"], state["meta"], m, k, n, dt, state["b"], c, stream=stream)
    elif kind == "sampled":
        with S.Plan.from_device(state["rowptr"], state["colidx"], m, k, state["colidx"].numel(), n, dt,
                                stream=stream) as plan:
            plan.run(state["values"], state["b"], c, stream=stream)
    else:
        state["plan"].run(state["values"], state["b"], c, stream=stream)
    return c


# ------------------------------------------------------------------ what it takes
def _entries(case):
    """Nonzeros of A: exactly for layers and training, else as expected."""
    kind = case["kind"]
    if kind in ("layer", "train_layer"):
        return max(1, round(case["m"] * case["k"] * case["density"]))
    if kind == "zipf":
        return case["total"]
    if kind == "sampled":
        return case["m"] * case["fanout"] * 0.9
    # distinct pairs (either direction) hit by `edges` R-MAT samples with both ids below `nodes`, and the loops:
    # cells counted by how many of their levels lie in the first and in the two mixed quadrants
    n, levels = case["nodes"], _levels(case["nodes"])
    a, b, c = RMAT
    d = 1 - a - b - c
    cells = {(True, True, 0, 0): 1}  # (u and v still on the last valid id's path, levels in each) -> cells
    for level in reversed(range(levels)):
        bit = (n - 1) >> level & 1
        nxt = {}
        for (tu, tv, i, j), count in cells.items():
            for bu in (0, 1):
                for bv in (0, 1):
                    if (tu and bu > bit) or (tv and bv > bit):
                        continue
                    key = (tu and bu == bit, tv and bv == bit, i + (bu + bv == 0), j + (bu + bv == 1))
                    nxt[key] = nxt.get(key, 0) + count
        cells = nxt
    prob = {key: a ** key[2] * b ** key[3] * d ** (levels - key[2] - key[3]) for key in cells}
    valid = sum(cells[key] * prob[key] for key in cells)
    pairs = sum(cells[key] * -math.expm1(-2.0 * case["edges"] / valid * prob[key]) for key in cells)
    return (n + pairs) * (0.9 if kind == "train_graph" else 1.0)


def work(case):
    kind, n, e = case["kind"], case["n"], SIZE[case["dtype"]]
    m, k = _shape(case)
    dense = k * n * e + m * n * 4
    if kind == "bell":
        nnz = m * k * case["density"]
        return {"bytes": int(nnz * e + nnz / case["block"] ** 2 * 4 + dense), "flops": int(2 * nnz * n)}
    if kind == "s24":
        return {"bytes": int(m * k * (e / 2 + 0.125) + dense), "flops": int(m * k * n)}
    nnz = _entries(case)
    forward = nnz * (4 + e) + 4 * (m + 1) + dense
    if not kind.startswith("train"):
        return {"bytes": int(forward), "flops": int(2 * nnz * n)}
    # backward: the gradient of C and B read once, both gradients written once
    backward = m * n * 4 + nnz * e + k * n * e
    return {"bytes": int(forward + backward), "flops": int(6 * nnz * n)}


def tolerance(case):
    if case["kind"].startswith("train") and case["dtype"] != "f32":
        # gradients leave in 16 bits
        return {"rel": 7e-3 if case["dtype"] == "bf16" else 8e-4}
    # fp32 sums: 1e-8 (short rows) to 2.8e-7 (the longest) from the 64-bit result, times four
    return {"rel": 1.2e-6}


def _sum_rows(rows, cols, values, b, m):
    """sum of values[j] * b[cols[j]] into row rows[j] (ascending), in 64 bits: running sums over a
    stretch of entries, differences at the ends of its rows."""
    n = b.shape[1]
    out = torch.zeros((m, n), dtype=torch.float64, device=DEV)
    step = max(1, (1 << 27) // n)
    for j in range(0, rows.numel(), step):
        r = rows[j:j + step]
        part = b[cols[j:j + step]].double()
        part *= values[j:j + step].double()[:, None]
        here, count = torch.unique_consecutive(r, return_counts=True)
        run = torch.cumsum(part.t().contiguous(), 1)[:, torch.cumsum(count, 0) - 1].t()
        run[1:] -= run[:-1].clone()
        out[here] += run
    return out


def exact(case, seed):
    if case["kind"] in ("bell", "s24"):
        a, b = _dense_inputs(case, seed)
        return a.double() @ b.double()
    rowptr, colidx, values, b, gc = _inputs(case, seed)
    m, k = _shape(case)
    rows, cols = _rows_of(rowptr), colidx.long()
    c = _sum_rows(rows, cols, values, b, m)
    if gc is None:
        return c
    gv = torch.empty(cols.numel(), dtype=torch.float64, device=DEV)
    step = max(1, (1 << 26) // case["n"])
    for j in range(0, cols.numel(), step):
        gv[j:j + step] = (gc[rows[j:j + step]].double() * b[cols[j:j + step]].double()).sum(1)
    by_col = torch.argsort(cols, stable=True)
    return {"c": c, "grad_values": gv, "grad_b": _sum_rows(cols[by_col], rows[by_col], values[by_col], gc, k)}
