"""The workloads that this engine's speed is measured on: y = alpha*A*x + beta*y
through its public entry points, over the matrix families, sizes, value types
and forms that its users run.

Matrices are made on the GPU from a seed (rows of distinct, ascending columns):

* ``banded``: row lengths N(mu, sigma) clipped to [min(8, mu), 400], columns
  spread over a window of +-hw around the diagonal, normal values -- finite
  element and finite difference meshes;
* ``rmat``: R-MAT (.57, .19, .19, .05) with ef edges a vertex, duplicates
  merged, cut to n vertices, values 1 -- web and social graphs;
* ``powerlaw``: row lengths p(L) ~ (L + 2.23)^-2 on [1, 2000], columns spread
  over all of x, uniform values.

A case names its operation (``op``): ``spmv`` and ``spmm`` are products of a
plan that the program keeps, ``batch`` a set of matrices replayed as one graph,
``dropin`` the reference's call on host arrays, which uploads the matrix,
analyses it, multiplies once and copies y back.
"""
import math

import numpy as np
import torch

DTYPES = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}
VAL_BYTES = {"f64": 8, "f32": 4, "bf16": 2}
RMAT = (0.57, 0.19, 0.19)
LMAX = 2000
SHIFT = 2.23


def _spmv(name, family, n, **more):
    case = {"name": name, "op": "spmv", "family": family, "n": n, "mu": 0.0, "sigma": 0.0, "hw": 0,
            "ef": 0, "dtype": "f64", "fmt": "csr", "kernel": 0, "k": 1, "chunks": 0,
            "part": "v1", "beta": 0.0}
    case.update(more)
    return case


def listed():
    return [
        # A small irregular system solved step by step: a launch's own cost counts.
        _spmv("spmv_powerlaw_20k_f64", "powerlaw", 20_000),
        # A 27-point stencil on a mid-sized 3-D mesh, the common structured solve.
        _spmv("spmv_stencil27_512k_f64", "banded", 512_000, mu=27.0, sigma=0.0, hw=6_500),
        # The large finite element matrix in eight chunks: the engine's headline workload.
        _spmv("spmv_banded_2m_f64", "banded", 2_000_000, mu=140.0, sigma=40.0, hw=50_000,
              chunks=8, part="v1_numa"),
        # The same with stored FP32 values, as preconditioners keep them.
        _spmv("spmv_banded_2m_f32", "banded", 2_000_000, mu=140.0, sigma=40.0, hw=50_000,
              dtype="f32", chunks=8, part="v1_numa"),
        # A large graph with an accumulated result (PageRank-like steps).
        _spmv("spmv_rmat22_f64", "rmat", 1 << 22, ef=17, beta=0.5),
        # A ragged mid-sized graph, edge weights in BF16.
        _spmv("spmv_rmat_1500k_bf16", "rmat", 1_500_001, ef=16, dtype="bf16"),
        # Eight vectors at once over the large graph (block methods, embeddings).
        _spmv("spmm8_rmat22_f64", "rmat", 1 << 22, op="spmm", k=8, ef=17),
        # Four right-hand sides of a mid-sized finite element system (block solvers).
        _spmv("spmm4_banded_400k_f64", "banded", 400_009, op="spmm", k=4, mu=140.0, sigma=40.0,
              hw=10_000),
        # The merge-path kernel (switch 2), asked for by name, on an irregular matrix.
        _spmv("merge_powerlaw_1m_f64", "powerlaw", 1_000_003, kernel=2),
        # The CSR5-style kernel (switch 3), asked for by name, on a graph.
        _spmv("csr5_rmat20_f64", "rmat", 1 << 20, ef=16, kernel=3),
        # Sixteen systems of uneven sizes, meshes and graphs in turn, one graph launch.
        {"name": "batch16_f32", "op": "batch", "count": 16, "n_lo": 10_000, "n_hi": 1_000_000,
         "dtype": "f32"},
        # The reference's own entry point on host arrays, one product a call.
        _spmv("dropin_powerlaw_20k_f64", "powerlaw", 20_000, op="dropin", kernel=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choices(["spmv", "spmm", "kernel", "batch", "dropin"], [8, 4, 3, 1, 2])[0]
    if op == "batch":
        lo = _log_int(rng, 5_000, 50_000)
        return {"op": "batch", "count": rng.randint(8, 16), "n_lo": lo,
                "n_hi": _log_int(rng, 4 * lo, 600_000), "dtype": rng.choice(["f64", "f32", "bf16"])}
    case = _spmv("", "banded", 0)
    del case["name"]
    case["family"] = rng.choice(["banded", "banded", "rmat", "powerlaw"])
    case["dtype"] = rng.choice(["f64", "f64", "f32", "bf16"])
    case["beta"] = rng.choice([0.0, 0.0, 0.5])
    case["op"] = "spmv" if op == "kernel" else op
    top = {"spmv": 1.0, "kernel": 0.5, "spmm": 0.25, "dropin": 0.02}[op]  # of the largest sizes
    if case["family"] == "banded":
        case["mu"] = round(math.exp(rng.uniform(math.log(4.0), math.log(140.0))), 1)
        case["sigma"] = round(case["mu"] * rng.choice([0.0, 0.1, 0.3]), 1)
        case["n"] = _log_int(rng, 5_000, max(20_000, min(4e6, top * 2e8 / case["mu"])))
        case["hw"] = max(int(2 * case["mu"]) + 8, case["n"] // rng.choice([400, 80, 40, 10]))
        case["chunks"] = rng.choice([0, 0, 8])
        case["part"] = "v1_numa" if case["chunks"] else "v1"
    elif case["family"] == "rmat":
        case["ef"] = rng.randint(8, 17)
        case["n"] = _log_int(rng, 5_000, max(20_000, top * 4e6))
    else:
        case["n"] = _log_int(rng, 2_000, max(20_000, top * 2e6))
    if op == "spmm":
        case["k"] = rng.choice([2, 4, 8, 16])
    elif op == "kernel":
        case["kernel"] = rng.choice([2, 2, 3, 3, 4])
        case["fmt"] = "coo" if case["kernel"] == 4 else "csr"
    elif op == "dropin":
        case["kernel"] = rng.choice([1, 1, 2, 3])
        case["dtype"] = "f64"
        case["beta"] = 0.0
    else:
        case["fmt"] = rng.choice(["csr", "csr", "csr", "coo", "csc"])
    return case


# ---- matrices --------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _row_ptr(lengths):
    rp = torch.zeros(lengths.numel() + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(lengths, 0, out=rp[1:])
    return rp


def _spread(lengths, first, width, g):
    """Row r's columns: one in each of lengths[r] equal parts of its window
    [first[r], first[r] + width[r]), so distinct and ascending."""
    rp = _row_ptr(lengths)
    nnz = int(rp[-1])
    row = torch.repeat_interleave(torch.arange(lengths.numel(), device="cuda", dtype=torch.int32),
                                  lengths, output_size=nnz)
    col = torch.empty(nnz, dtype=torch.int32, device="cuda")
    step = 1 << 26
    for a in range(0, nnz, step):
        b = min(a + step, nnz)
        r = row[a:b].long()
        j = torch.arange(a, b, device="cuda") - rp[r]
        w, length = width[r], lengths[r]
        lo = j * w // length
        part = (j + 1) * w // length - lo
        u = torch.rand(b - a, device="cuda", generator=g)
        col[a:b] = (first[r] + lo + torch.minimum((u * part).long(), part - 1)).int()
    return rp.int(), row, col


def _banded(n, mu, sigma, hw, g):
    lengths = torch.full((n,), mu, device="cuda")
    if sigma > 0:
        lengths += sigma * torch.randn(n, device="cuda", generator=g)
    lengths = lengths.round().clamp(min(8.0, max(1.0, round(mu))), 400.0).long()
    r = torch.arange(n, device="cuda")
    first = (r - hw).clamp(min=0)
    width = (r + hw).clamp(max=n - 1) - first + 1
    rp, row, col = _spread(torch.minimum(lengths, width), first, width, g)
    return rp, row, col, torch.randn(col.numel(), device="cuda", generator=g, dtype=torch.float64)


def _powerlaw_weights(n):
    w = (np.arange(1, min(LMAX, n) + 1) + SHIFT) ** -2.0
    return w / w.sum()


def _powerlaw(n, g):
    cdf = torch.from_numpy(np.cumsum(_powerlaw_weights(n))).to("cuda")
    u = torch.rand(n, device="cuda", generator=g, dtype=torch.float64)
    lengths = torch.searchsorted(cdf, u).clamp(max=cdf.numel() - 1) + 1
    zero = torch.zeros(n, dtype=torch.int64, device="cuda")
    rp, row, col = _spread(lengths, zero, zero + n, g)
    val = 2.0 * torch.rand(col.numel(), device="cuda", generator=g, dtype=torch.float64) - 1.0
    return rp, row, col, val


def _rmat(n, ef, g):
    scale = max(1, (n - 1).bit_length())
    edges = ef << scale
    a, b, c = RMAT
    row = torch.zeros(edges, dtype=torch.int32, device="cuda")
    col = torch.zeros(edges, dtype=torch.int32, device="cuda")
    for _ in range(scale):
        u = torch.rand(edges, device="cuda", generator=g)
        row.mul_(2).add_(u >= a + b)
        col.mul_(2).add_(((u >= a) & (u < a + b)) | (u >= a + b + c))
    keys = row.long().mul_(n).add_(col)
    if n != 1 << scale:
        keys = keys[(row < n) & (col < n)]
    del row, col, u
    keys = torch.unique(keys)
    row = (keys // n).int()
    col = (keys % n).int()
    rp = _row_ptr(torch.bincount(row, minlength=n)).int()
    return rp, row, col, torch.ones(col.numel(), device="cuda", dtype=torch.float64)


def _matrix(case, g):
    """(row_ptr, row of each element, col, val); val of the case's value type."""
    if case["family"] == "banded":
        rp, row, col, val = _banded(case["n"], case["mu"], case["sigma"], case["hw"], g)
    elif case["family"] == "rmat":
        rp, row, col, val = _rmat(case["n"], case["ef"], g)
    else:
        rp, row, col, val = _powerlaw(case["n"], g)
    return rp, row, col, val.to(DTYPES[case["dtype"]])


def _vectors(case, g):
    shape = (case["n"],) if case["k"] == 1 else (case["n"], case["k"])
    x = 2.0 * torch.rand(shape, device="cuda", generator=g, dtype=torch.float64) - 1.0
    y = 2.0 * torch.rand(shape, device="cuda", generator=g, dtype=torch.float64) - 1.0
    return x, y


def _batch_cases(case):
    """The batch's matrices: sizes spread evenly over the logarithm of the
    range, a mesh and a graph in turn."""
    out = []
    for i in range(case["count"]):
        n = int(round(case["n_lo"] * (case["n_hi"] / case["n_lo"]) ** (i / (case["count"] - 1))))
        more = ({"family": "banded", "mu": 140.0, "sigma": 40.0, "hw": min(50_000, n // 40)}
                if i % 2 == 0 else {"family": "rmat", "ef": 16})
        out.append(_spmv("", n=n, dtype=case["dtype"], **more))
    return out


# ---- one pass ----------------------------------------------------------------------

def prepare(case, seed):
    from hpda_sblas_pnnl_amd import SpmvBatch, SpmvPlan

    g = _generator(seed)
    if case["op"] == "batch":
        items = []
        for c in _batch_cases(case):
            rp, _, col, val = _matrix(c, g)
            x, y = _vectors(c, g)
            items.append({"m": c["n"], "n": c["n"], "row_ptr": rp, "col": col, "val": val,
                          "x": x, "y": y})
        return {"op": "batch", "batch": SpmvBatch(items), "y": [it["y"] for it in items]}
    rp, row, col, val = _matrix(case, g)
    x, y = _vectors(case, g)
    n = case["n"]
    if case["op"] == "dropin":
        return {"op": "dropin", "n": n, "kernel": case["kernel"],
                "arrays": [t.cpu().numpy() for t in (val, rp, col, x)], "y": y.cpu().numpy()}
    a0, a1 = rp, col
    if case["fmt"] == "coo":
        a0 = row
    elif case["fmt"] == "csc":
        order = torch.sort(col, stable=True).indices
        a0 = _row_ptr(torch.bincount(col, minlength=n)).int()
        a1, val = row[order], val[order]
    plan = SpmvPlan(case["fmt"], n, n, a0, a1, val, kernel=case["kernel"], chunks=case["chunks"],
                    part_mode=case["part"])
    return {"op": case["op"], "plan": plan, "x": x, "y": y, "beta": case["beta"]}


def run(state):
    if state["op"] == "batch":
        state["batch"].graph_launch()
        return state["y"]
    if state["op"] == "dropin":
        from hpda_sblas_pnnl_amd import spMV_mgpu_v1
        val, rp, col, x = state["arrays"]
        spMV_mgpu_v1(state["n"], state["n"], len(val), 1.0, val, rp, col, x, 0.0, state["y"], 1,
                     state["kernel"])
        return state["y"]
    product = state["plan"].spmm if state["op"] == "spmm" else state["plan"].spmv
    return product(state["x"], state["y"], 1.0, state["beta"])


# ---- what a pass needs -----------------------------------------------------------

def _rmat_kept(n):
    """Share of R-MAT edges with both ends below n: bit by bit from the top,
    for pairs of prefixes that are below or still equal to those of n."""
    scale = max(1, (n - 1).bit_length())
    if n == 1 << scale:
        return 1.0
    p = {(0, 0): RMAT[0], (0, 1): RMAT[1], (1, 0): RMAT[2], (1, 1): 1.0 - sum(RMAT)}
    state = {(True, True): 1.0}  # prefix equal to n's: (row, col)
    for bit in range(scale - 1, -1, -1):
        want, after = (n >> bit) & 1, {}
        for (er, ec), share in state.items():
            for (br, bc), q in p.items():
                if (er and br > want) or (ec and bc > want):
                    continue
                key = (er and br == want, ec and bc == want)
                after[key] = after.get(key, 0.0) + share * q
        state = after
    return state.get((False, False), 0.0)


def _elements(case):
    """Elements of the case's matrix: its mean, R-MAT's before duplicates merge."""
    n = case["n"]
    if case["family"] == "banded":
        return n * case["mu"]
    if case["family"] == "rmat":
        return (case["ef"] << max(1, (n - 1).bit_length())) * _rmat_kept(n)
    w = _powerlaw_weights(n)
    return n * float((w * np.arange(1, len(w) + 1)).sum())


def work(case):
    """The matrix read once in its own format (4-byte indices, values as
    stored), x read once, y written once and read where beta is not 0; two
    operations an element and vector."""
    if case["op"] == "batch":
        parts = [work(c) for c in _batch_cases(case)]
        return {key: sum(p[key] for p in parts) for key in ("bytes", "flops")}
    n, k, nnz = case["n"], case["k"], _elements(case)
    index = 4.0 * nnz if case["fmt"] == "coo" else 4.0 * (n + 1)
    vectors = 8.0 * n * k * (3 if case["beta"] else 2)
    return {"bytes": nnz * (VAL_BYTES[case["dtype"]] + 4.0) + index + vectors,
            "flops": 2.0 * nnz * k}


def _product(rp, row, col, val, x, y, beta):
    out = torch.zeros_like(y)
    step = (1 << 26) // (1 if x.dim() == 1 else x.shape[1])
    for a in range(0, col.numel(), step):
        c, v = col[a:a + step].long(), val[a:a + step].double()
        out.index_add_(0, row[a:a + step], x[c] * (v if x.dim() == 1 else v[:, None]))
    return out + beta * y if beta else out


def exact(case, seed):
    g = _generator(seed)
    if case["op"] == "batch":
        out = []
        for c in _batch_cases(case):
            matrix = _matrix(c, g)
            out.append(_product(*matrix, *_vectors(c, g), 0.0))
        return out
    matrix = _matrix(case, g)
    return _product(*matrix, *_vectors(case, g), case["beta"])
