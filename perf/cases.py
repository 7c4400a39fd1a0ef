"""Performance cases of the SpMM operator: what its users have it do, over the range of sizes and types they use.

A case names a matrix family, its size, an element type and a feature dimension N; one pass is C = A * B through
`Plan.run` with the plan, B and C resident on the GPU (family "convert": from CSR arrays on the host through the
tile converter and a new plan to C).  Families, as in hopper_spmm_amd/generators.py:

  uniform   entries drawn uniformly, `per_row` a row: sparse solvers, sampled interactions
  graph     R-MAT adjacency (power-law degrees, values 1 / out-degree): message passing, power iteration
  pruned    dense weight of which the fraction `keep` of largest magnitude is kept: unstructured sparse layers
  block     weight kept in 16 x 16 squares with probability `keep`: block-sparse layers
  convert   a graph that arrives as CSR on the host and is multiplied once: new adjacency per batch

N small is the decode side of a layer (a few tokens), or a graph's classes, or a single vector; N large the
prefill side and hidden features.  Inputs are made on the GPU from the seed alone.
"""
import math

import numpy as np
import torch

import hopper_spmm_amd as hs

DTYPES = {"fp16": (hs.FP16, torch.float16, 2), "bf16": (hs.BF16, torch.bfloat16, 2), "fp32": (hs.TF32, torch.float32, 4)}
BLOCK = 16
RMAT = (0.57, 0.19, 0.19, 0.05)


def _case(family, rows, cols, amount, dtype, n, tiles="plain"):
    """amount: entries per row (uniform), edges per vertex (graph, convert), kept fraction (pruned, block)."""
    return {"family": family, "rows": rows, "cols": cols, "amount": amount, "dtype": dtype, "n": n, "tiles": tiles}


def listed():
    return [
        # a small operator applied over and over: launch latency
        dict(_case("uniform", 4096, 4096, 41.0, "fp16", 64), name="uniform_small"),
        # interactions without any locality
        dict(_case("uniform", 65536, 65536, 16.0, "fp16", 128), name="uniform_sparse"),
        # message passing on a million-vertex graph, hidden features
        dict(_case("graph", 1 << 20, 1 << 20, 16.0, "fp16", 128), name="graph_large"),
        # full-precision features of a data set: neither a power of two of vertices nor of features
        dict(_case("graph", 150001, 150001, 16.0, "fp32", 100, "bitmap"), name="graph_fp32"),
        # the last layer of a graph network: a few classes
        dict(_case("graph", 262144, 262144, 16.0, "bf16", 16), name="graph_narrow"),
        # power iteration: one vector
        dict(_case("graph", 500000, 500000, 12.0, "fp16", 1), name="graph_vector"),
        # unstructured sparse layer kept in fp32
        dict(_case("pruned", 11008, 4096, 0.10, "fp32", 256), name="pruned_fp32"),
        # the same kind of layer while decoding a small batch
        dict(_case("pruned", 4096, 11008, 0.10, "bf16", 16), name="pruned_decode"),
        # odd shapes: a layer less pruned, a ragged number of tokens
        dict(_case("pruned", 5003, 3001, 0.20, "bf16", 333), name="pruned_ragged"),
        # block-sparse layer, decode and prefill
        dict(_case("block", 4096, 14336, 0.50, "fp16", 16), name="block_decode"),
        dict(_case("block", 4096, 14336, 0.50, "fp16", 512), name="block_prefill"),
        # a graph seen once: conversion, plan, product
        dict(_case("convert", 262144, 262144, 16.0, "fp16", 128), name="convert_graph"),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _size(rng, low, high, step):
    """A size between low and high, spread over its logarithm; half of the time a multiple of `step`."""
    v = _log(rng, low, high)
    return max(low, v - v % step) if rng.random() < 0.5 and v >= step else v


def _draw_family(rng):
    family = rng.choice(["uniform", "uniform", "graph", "graph", "graph", "pruned", "pruned", "pruned", "block", "block",
                         "convert"])
    dtype = rng.choice(["fp16", "bf16", "fp32"])
    n = _size(rng, 1, 1024, 16)
    if family == "uniform":
        rows, cols = _size(rng, 2048, 131072, 256), _size(rng, 2048, 131072, 256)
        return _case(family, rows, cols, float(_log(rng, 4, 256)), dtype, n)
    if family in ("graph", "convert"):
        vertices = _size(rng, 8192, (1 << 20) if family == "graph" else (1 << 18), 4096)
        return _case(family, vertices, vertices, float(_log(rng, 4, 32)), dtype, n, rng.choice(["plain", "plain", "bitmap"]))
    rows, cols = _size(rng, 1024, 16384, 256), _size(rng, 1024, 16384, 256)
    keep = math.exp(rng.uniform(math.log(0.03), math.log(0.30))) if family == "pruned" else rng.uniform(0.2, 0.6)
    return _case(family, rows, cols, round(keep, 4), dtype, n)


def draw(rng):
    """One more case of these ranges; none costs more than the largest listed one of its kind."""
    while True:
        c = _draw_family(rng)
        nnz = _expected_nnz(c)
        gathered, products = nnz * c["n"] * DTYPES[c["dtype"]][2], nnz * c["n"]
        if c["family"] in ("pruned", "block"):
            fits = c["rows"] * c["cols"] <= 4096 * 14336 and products <= 15.1e9
            fits = fits and (c["dtype"] != "fp32" or products <= 7.5e9)
        elif c["family"] == "convert":
            fits = nnz <= 4.0e6 and gathered <= 1.1e9
        else:
            fits = nnz <= 16.1e6 and gathered <= 4.2e9
        if fits and _shape_known(c):
            return c


def _shape_known(c):
    """At least one entry for every eight rows: a matrix, not a handful of entries."""
    return _expected_nnz(c) * 8 >= c["rows"]


# ---- inputs -------------------------------------------------------------------------------------------------


def _uniform_keys(c, gen):
    count = int(c["rows"] * c["amount"])
    r = torch.randint(c["rows"], (count,), generator=gen, device="cuda")
    k = torch.randint(c["cols"], (count,), generator=gen, device="cuda")
    return torch.unique(r * c["cols"] + k)


def _graph_keys(c, gen):
    a, b, cc, _ = RMAT
    nv, count = c["rows"], int(c["rows"] * c["amount"])
    scale = max(1, (nv - 1).bit_length())
    r = torch.zeros(count, dtype=torch.int64, device="cuda")
    k = torch.zeros(count, dtype=torch.int64, device="cuda")
    for _ in range(scale):
        u = torch.rand(count, generator=gen, device="cuda")
        low = u >= a + b
        right = ((u >= a) & ~low) | (u >= a + b + cc)
        r, k = (r << 1) | low, (k << 1) | right
    if nv != 1 << scale:                    # the 2^scale ids squeezed into nv, in order
        r, k = (r * nv) >> scale, (k * nv) >> scale
    return torch.unique(r * nv + k)


def _csr(c, seed):
    """The matrix as CSR on the host (values as the framework stores them)."""
    rows, cols = c["rows"], c["cols"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 2 + 1)
    if c["family"] == "uniform":
        keys = _uniform_keys(c, gen)
        values = torch.rand(keys.numel(), generator=gen, device="cuda") * 2.0 - 1.0
    elif c["family"] in ("graph", "convert"):
        keys = _graph_keys(c, gen)
        values = None
    elif c["family"] == "pruned":
        w = torch.randn(rows * cols, generator=gen, device="cuda") * 0.02
        kept = max(1, int(round(rows * cols * c["amount"])))
        threshold = torch.kthvalue(w.abs(), rows * cols - kept + 1).values
        keys = torch.nonzero(w.abs() >= threshold).flatten()
        values = w[keys]
    else:
        br, bc = -(-rows // BLOCK), -(-cols // BLOCK)
        keep = torch.rand((br, bc), generator=gen, device="cuda") < c["amount"]
        keep[0, 0] = True
        mask = keep.repeat_interleave(BLOCK, 0)[:rows].repeat_interleave(BLOCK, 1)[:, :cols]
        keys = torch.nonzero(mask.flatten()).flatten()
        values = torch.randn(keys.numel(), generator=gen, device="cuda") * 0.02
    r = torch.div(keys, cols, rounding_mode="floor")
    counts = torch.bincount(r, minlength=rows)
    if values is None:
        values = 1.0 / counts[r].float()
    row_ptr = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
    row_ptr[1:] = torch.cumsum(counts, 0)
    stored = values.to(DTYPES[c["dtype"]][1])
    host = stored.cpu() if stored.dtype == torch.float32 else stored.view(torch.int16).cpu()
    host = host.numpy() if stored.dtype == torch.float32 else host.numpy().view(np.uint16)
    return {"row_ptr": row_ptr.int().cpu().numpy().view(np.uint32),
            "col_idx": (keys - r * cols).int().cpu().numpy().view(np.uint32), "values": host}


def _convert(c, csr):
    make = hs.csr_to_bitmap if c["tiles"] == "bitmap" else hs.csr_to_btcf
    return make(c["rows"], c["cols"], csr["row_ptr"], csr["col_idx"], csr["values"], DTYPES[c["dtype"]][0])


def prepare(case, seed):
    csr = _csr(case, seed)
    dtype = DTYPES[case["dtype"]][1]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 2)
    state = {"case": case, "n": case["n"],
             "B": torch.randn((case["cols"], case["n"]), generator=gen, device="cuda").to(dtype),
             "C": torch.empty((case["rows"], case["n"]), dtype=dtype, device="cuda")}
    if case["family"] == "convert":
        state["csr"] = csr
    else:
        state["plan"] = hs.Plan(_convert(case, csr))
    return state


def run(state):
    B, C, n = state["B"], state["C"], state["n"]
    stream = torch.cuda.current_stream().cuda_stream
    if "plan" in state:
        state["plan"].run(B.data_ptr(), C.data_ptr(), n, stream)
        return C
    matrix = _convert(state["case"], state["csr"])
    plan = hs.Plan(matrix)
    plan.run(B.data_ptr(), C.data_ptr(), n, stream)
    plan.close()
    return C


# ---- what a pass cannot do without -----------------------------------------------------------------------------


def _rmat_expected(c):
    """Expected numbers of distinct edges and of columns with an edge (the ids are 2^scale before they are squeezed)."""
    a, b, cc, d = RMAT
    scale, draws = max(1, (c["rows"] - 1).bit_length()), c["rows"] * c["amount"]
    squeeze = (1 << scale) / c["rows"]      # ids that share a vertex
    edges = 0.0
    for i in range(scale + 1):
        for j in range(scale + 1 - i):
            for k in range(scale + 1 - i - j):
                m = scale - i - j - k
                cells = math.comb(scale, i) * math.comb(scale - i, j) * math.comb(scale - i - j, k)
                hit = draws * a ** i * b ** j * cc ** k * d ** m * squeeze ** 2
                edges += cells / squeeze ** 2 * -math.expm1(-hit)
    cols = sum(math.comb(scale, i) / squeeze * -math.expm1(-draws * squeeze * (a + cc) ** i * (b + d) ** (scale - i))
               for i in range(scale + 1))
    return edges, cols


def _expected_nnz(c):
    cells = float(c["rows"]) * c["cols"]
    if c["family"] == "uniform":
        return cells * -math.expm1(-c["rows"] * c["amount"] / cells)
    if c["family"] in ("graph", "convert"):
        return _rmat_expected(c)[0]
    return cells * c["amount"]


def work(case):
    """Every stored entry and its place read once, every row of B that an entry names, every element of C written.
    A place is four bytes, or one bit for every element of the matrix where that is less; a block has one place."""
    size, n = DTYPES[case["dtype"]][2], case["n"]
    nnz, used, cells = _expected_nnz(case), float(case["cols"]), float(case["rows"]) * case["cols"]
    if case["family"] in ("graph", "convert"):
        used = _rmat_expected(case)[1]
    elif case["family"] == "uniform":
        used *= -math.expm1(-nnz / case["cols"])
    places = nnz / BLOCK ** 2 if case["family"] == "block" else nnz
    entries = nnz * size + min(4.0 * places, cells / 8.0) + 4.0 * (case["rows"] + 1)
    total = entries + size * n * (used + case["rows"])
    if case["family"] == "convert":         # the entries once more as tiles, at least their values and columns
        total += entries
    return {"bytes": total, "flops": 2.0 * nnz * n}


def tolerance(case):
    """Two sums of exact products in another order, rounded once to the element type.  fp32 storage: layers go through
    products of bf16 high and low parts (16 bits of each factor kept), the rest through fp32 products."""
    if case["dtype"] == "fp16":
        return {"rel": 1e-3, "max": 1e-2}
    if case["dtype"] == "bf16":
        return {"rel": 8e-3, "max": 4e-2}
    if case["family"] in ("graph", "convert"):
        return {"rel": 1e-5, "max": 1e-3}
    return {"rel": 4e-5, "max": 1e-3}
