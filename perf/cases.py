"""What the speed of this framework is measured on: the calls that its users make, over the sizes that they make
them at.

    listed()              the cases
    draw(rng)             one more case of the same ranges
    prepare(case, seed)   what a program has in hand before the call (inputs on the GPU, the decomposed matrix)
    run(state)            one pass through the public entry points, and its outputs
    work(case)            the bytes and operations that a pass cannot do without
    tolerance(case)       how far the outputs of two correct implementations may lie apart

A case names an operation ("op"), a sparsity pattern ("pattern": rows x cols, "degree" nonzeros per row) and the dense
side ("k" elements per dense row, "dtype", and for attention "heads").  The patterns are those of the five benchmark
configurations (rode_amd/workloads.py) drawn on the GPU, so that fresh inputs are quick to make."""
import math

import torch

from rode_amd import RoDeCSR, rode_sddmm, rode_spmm, sparse_attention
from rode_amd import rode_sddmm_hip

DTYPES = {"f32": torch.float32, "f16": torch.float16, "f64": torch.float64}
BYTES = {"f32": 4, "f16": 2, "f64": 8}

STRETCH = 6          # power law: degree = STRETCH * (Zipf(2.1) - 1) + U{1..STRETCH}
POWER_LAW_MEAN = 24  # ... and what that averages over a large matrix
HUB_MOST = 200_000   # ... and its largest degree
SIGMA = 1.5          # lognormal degrees
ROW_MOST = 20_000    # ... and their largest


def listed():
    return [
        # Many small matrices, or one small matrix many times: the smallest size of the op's own comparison with torch.
        # Launches and host work decide.
        {"name": "sddmm_small", "op": "sddmm", "pattern": "uniform", "rows": 1024, "cols": 1024, "degree": 64, "k": 32, "dtype": "f32"},
        # The first benchmark configuration: one percent of a 4096 x 4096 matrix.
        {"name": "spmm_small", "op": "spmm", "pattern": "uniform", "rows": 4096, "cols": 4096, "degree": 41, "k": 32, "dtype": "f32"},
        # The odd, non-square size of the same comparison.
        {"name": "sddmm_odd", "op": "sddmm", "pattern": "uniform", "rows": 4093, "cols": 4099, "degree": 128, "k": 128, "dtype": "f32"},
        # Message passing over a middle-sized graph with ragged rows (second configuration), inference.
        {"name": "spmm_graph", "op": "spmm", "pattern": "lognormal", "rows": 65536, "cols": 65536, "degree": 16, "k": 128, "dtype": "f32"},
        # A training step of a graph convolution: the product and its gradient (a product with the transpose).
        {"name": "graph_train", "op": "spmm_train", "pattern": "lognormal", "rows": 100_003, "cols": 100_003, "degree": 16, "k": 64, "dtype": "f32"},
        # Edge scores on a FEM-like mesh (third configuration): every row short.
        {"name": "sddmm_band", "op": "sddmm", "pattern": "banded", "rows": 1_000_000, "cols": 1_000_000, "degree": 27, "band": 256, "k": 128, "dtype": "f32"},
        # A mesh operator applied to a block of vectors in double precision, as solvers do.
        {"name": "spmm_band_f64", "op": "spmm", "pattern": "banded", "rows": 500_000, "cols": 500_000, "degree": 27, "band": 256, "k": 32, "dtype": "f64"},
        # The headline: a power-law graph with hubs of up to 200 000 neighbours (fourth configuration).
        {"name": "spmm_powerlaw", "op": "spmm", "pattern": "powerlaw", "rows": 2_000_000, "cols": 2_000_000, "degree": POWER_LAW_MEAN, "k": 128, "dtype": "f32"},
        # Edge scores on the same graph from half-precision features.
        {"name": "sddmm_powerlaw_f16", "op": "sddmm", "pattern": "powerlaw", "rows": 2_000_000, "cols": 2_000_000, "degree": POWER_LAW_MEAN, "k": 64, "dtype": "f16"},
        # A layer of sparse attention at inference: sliding window and random columns (fifth configuration), eight heads.
        {"name": "attention_heads_f16", "op": "attention", "pattern": "mask", "rows": 16384, "cols": 16384, "window": 512, "extra": 64, "k": 64, "dtype": "f16", "heads": 8},
        # The same mask in training, one head in single precision: forward and backward.
        {"name": "attention_train", "op": "attention_train", "pattern": "mask", "rows": 16384, "cols": 16384, "window": 512, "extra": 64, "k": 64, "dtype": "f32", "heads": 1},
        # A new graph arrives (sampled subgraphs, dynamic masks): decomposition and plan, before any product.
        {"name": "build_graph", "op": "build", "pattern": "lognormal", "rows": 65536, "cols": 65536, "degree": 16, "k": 128, "dtype": "f32"},
    ]


def _spread(rng, low, high):
    """A size between low and high, spread over its logarithm; odd ones among them."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["small", "small", "graph", "graph", "banded", "powerlaw", "mask", "mask", "build"])
    if kind == "small":
        rows = _spread(rng, 512, 16384)
        case = {"op": rng.choice(["spmm", "sddmm"]), "pattern": "uniform", "rows": rows, "cols": max(512, int(rows * rng.uniform(0.7, 1.4))),
                "degree": _spread(rng, 8, 128), "k": rng.choice([32, 48, 64, 96, 128]), "dtype": rng.choice(["f32", "f32", "f16"])}
    elif kind == "graph":
        rows = _spread(rng, 16384, 400_000)
        case = {"op": rng.choice(["spmm", "sddmm", "spmm_train", "spmm_train"]), "pattern": "lognormal", "rows": rows, "cols": rows,
                "degree": _spread(rng, 8, 32), "k": rng.choice([32, 64, 96, 128]), "dtype": rng.choice(["f32", "f32", "f16"])}
    elif kind == "banded":
        rows = _spread(rng, 50_000, 1_000_000)
        op = rng.choice(["spmm", "sddmm"])
        dtype = rng.choice(["f32", "f16", "f64"] if op == "spmm" else ["f32", "f16"])
        case = {"op": op, "pattern": "banded", "rows": rows, "cols": rows, "degree": rng.randint(9, 27), "band": rng.choice([128, 192, 256]),
                "k": 32 if dtype == "f64" else rng.choice([32, 64, 128]), "dtype": dtype}
    elif kind == "powerlaw":
        rows = _spread(rng, 200_000, 2_000_000)
        case = {"op": rng.choice(["spmm", "sddmm"]), "pattern": "powerlaw", "rows": rows, "cols": rows, "degree": POWER_LAW_MEAN,
                "k": rng.choice([32, 64, 128]), "dtype": rng.choice(["f32", "f16"])}
    elif kind == "mask":
        op = rng.choice(["attention", "attention_train"])
        case = {"op": op, "pattern": "mask", "rows": _spread(rng, 2048, 20_000), "window": 2 * _spread(rng, 64, 320), "extra": rng.choice([0, 16, 32, 64, 96]),
                "k": rng.choice([32, 64, 128]), "dtype": rng.choice(["f32", "f16"])}
        case["cols"] = case["rows"]
        # as many heads as stay below the work of the eight heads (one in training) listed above, sixteen at most
        room = 16384 * 576 * 64 * (8 if op == "attention" else 3) // (case["rows"] * (case["window"] + case["extra"]) * case["k"])
        case["heads"] = max(1, min(16, room, rng.choice([1, 2, 4, 8, 16])))
    else:
        rows = _spread(rng, 16384, 400_000)
        case = {"op": "build", "pattern": rng.choice(["lognormal", "uniform"]), "rows": rows, "cols": rows, "degree": _spread(rng, 8, 32), "k": 64, "dtype": "f32"}
    return case


# ---- inputs -----------------------------------------------------------------------------

def _lengths(case, gen, device):
    """Row lengths of a ragged pattern: the same for every seed but for where they start, so that the outputs of two
    seeds have the same shapes.  (Rotated by a multiple of four nonzeros: the decomposition works on slots aligned to
    four, and every row keeps its alignment.)"""
    rows, cols, pattern = case["rows"], case["cols"], case["pattern"]
    fixed = torch.Generator(device=device)
    fixed.manual_seed(1000 + rows)
    if pattern == "uniform":  # every position with the same probability
        lengths = torch.poisson(torch.full((rows,), float(case["degree"]), device=device), generator=fixed).long()
    elif pattern == "lognormal":
        normal = torch.randn(rows, generator=fixed, device=device)
        lengths = torch.exp(math.log(case["degree"]) - 0.5 * SIGMA * SIGMA + SIGMA * normal).long().clamp_(max=ROW_MOST)
    else:  # power law
        share = torch.arange(1, HUB_MOST // STRETCH + 2, device=device, dtype=torch.float64).pow(-2.1).cumsum(0)
        uniform = torch.rand(rows, generator=fixed, device=device, dtype=torch.float64)
        zipf = torch.searchsorted(share / share[-1], uniform)  # (minus one: the smallest is 0)
        lengths = (STRETCH * zipf + torch.randint(1, STRETCH + 1, (rows,), generator=fixed, device=device)).clamp_(max=HUB_MOST)
    lengths.clamp_(max=cols // 2)
    lengths[-1] += -int(lengths.sum()) % 4
    starts = lengths.cumsum(0) - lengths
    aligned = (starts % 4 == 0).nonzero().flatten()
    pick = int(torch.randint(0, aligned.numel(), (1,), generator=gen, device=device))
    return lengths.roll(-int(aligned[pick]))


def _distinct(gen, device, lengths, cols):
    """Sorted keys row * cols + column: for every row as many distinct columns as it is long, out of the first `cols`
    (an int, or one per row).  A sorted draw with repetition out of cols - length + 1 columns becomes one without when
    its i-th column moves up by i."""
    row = torch.repeat_interleave(torch.arange(lengths.numel(), device=device), lengths)
    room = (cols - lengths + 1)[row] if torch.is_tensor(cols) else cols - lengths[row] + 1
    stride = int(cols.max()) if torch.is_tensor(cols) else cols
    column = torch.rand(row.numel(), generator=gen, device=device, dtype=torch.float64).mul_(room).long()
    keys = torch.sort(column.add_(row * stride))[0]
    return keys.add_(torch.arange(row.numel(), device=device) - (lengths.cumsum(0) - lengths)[row]), row, stride


def _pattern(case, gen, device):
    """(row offsets on the CPU, columns, values) of the case's matrix, columns ascending within a row."""
    rows, cols, pattern = case["rows"], case["cols"], case["pattern"]
    if pattern == "banded":
        # `degree` of the `band` columns around the diagonal, every choice equally likely: column after column
        # is taken with probability (still wanted) / (still to come)
        band = case["band"]
        wanted = torch.full((rows,), float(case["degree"]), device=device)
        taken = torch.empty(band, rows, dtype=torch.bool, device=device)
        for t in range(band):
            taken[t] = torch.rand(rows, generator=gen, device=device) * (band - t) < wanted
            wanted -= taken[t].float()
        at = taken.t().nonzero()
        first = (torch.arange(rows, device=device) - band // 2).clamp_(0, cols - band)
        keys = at[:, 0] * cols + first[at[:, 0]] + at[:, 1]
    elif pattern == "mask":  # a sliding window, and random columns outside it
        half = case["window"] // 2
        row = torch.arange(rows, device=device)
        window = row[:, None] + torch.arange(-half, half, device=device)[None, :]
        keys = (row[:, None] * cols + window)[(window >= 0) & (window < cols)]
        if case["extra"]:
            low, high = (row - half).clamp_(min=0), (row + half).clamp_(max=cols)
            extra, at, stride = _distinct(gen, device, torch.full((rows,), case["extra"], device=device), cols - (high - low))
            column = extra - at * stride
            column += torch.where(column >= low[at], (high - low)[at], 0)
            keys = torch.sort(torch.cat([keys, at * cols + column]))[0]
    else:
        keys = _distinct(gen, device, _lengths(case, gen, device), cols)[0]
    offsets = torch.searchsorted(keys, torch.arange(rows + 1, device=device) * cols).to(torch.int32)
    columns = (keys % cols).to(torch.int32)
    if pattern == "powerlaw":  # mean over the neighbours
        lengths = offsets[1:] - offsets[:-1]
        values = torch.repeat_interleave(1.0 / lengths.clamp(min=1).float(), lengths)
    elif pattern == "mask":
        values = torch.ones(columns.numel(), device=device)
    else:
        values = torch.rand(columns.numel(), generator=gen, device=device) * 2 - 1
    return offsets.cpu(), columns, values


def prepare(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    rows, cols, k, dtype = case["rows"], case["cols"], case["k"], DTYPES[case["dtype"]]
    offsets, columns, values = _pattern(case, gen, device)
    state = {"op": case["op"]}
    if case["op"] == "build":
        state["args"] = (offsets, columns, values, device, rows, cols, k)
        return state

    def dense(*shape):
        return torch.randn(*shape, generator=gen, device=device, dtype=torch.float64 if dtype == torch.float64 else torch.float32).to(dtype)

    state["matrix"] = RoDeCSR(offsets, columns, values, device, rows, cols, k, config="auto")
    if case["op"] == "sddmm":
        state["lhs"], state["rhs"] = dense(rows, k), dense(cols, k)
    elif case["op"] == "spmm":
        if dtype == torch.float64:
            state["matrix"] = state["matrix"].with_values(values.double())
        state["dense"] = dense(cols, k)
    elif case["op"] == "spmm_train":
        state["dense"] = dense(cols, k).requires_grad_()
        state["grad"] = torch.randn(rows, k, generator=gen, device=device)
    else:
        lead = (case["heads"],) if case["heads"] > 1 else ()
        train = case["op"] == "attention_train"
        state["qkv"] = tuple(dense(*lead, n, k).requires_grad_(train) for n in (rows, cols, cols))
        if train:
            state["grad"] = torch.randn(*lead, rows, k, generator=gen, device=device)
    return state


def run(state):
    op = state["op"]
    if op == "build":
        matrix = RoDeCSR(*state["args"], config="auto")
        return {"block": matrix.block_indices, "start": matrix.st_offsets, "residue": matrix.residue_indices, "m1": matrix.m1, "m2": matrix.m2}
    matrix = state["matrix"]
    if op == "sddmm":
        return rode_sddmm(matrix, state["lhs"], state["rhs"])
    if op == "spmm":
        if state["dense"].dtype == torch.float64:  # (the op takes float32 and float16; double goes through the module's function)
            return rode_sddmm_hip.spmm_forward(matrix.block_indices, matrix.residue_indices, matrix.st_offsets, matrix.m1, matrix.m2, matrix.row_offsets,
                                               matrix.column_indices, matrix.values, matrix.m, matrix.n, state["dense"], plan=matrix.plan)
        return rode_spmm(matrix, state["dense"])
    if op == "spmm_train":
        out = rode_spmm(matrix, state["dense"])
        return (out,) + torch.autograd.grad(out, (state["dense"],), state["grad"])
    q, k, v = state["qkv"]
    out = sparse_attention(matrix, q, k, v)
    if op == "attention":
        return out
    return (out,) + torch.autograd.grad(out, (q, k, v), state["grad"])


# ---- what a pass cannot do without ---------------------------------------------------------

def _nonzeros(case):
    if case["pattern"] == "mask":
        half = case["window"] // 2
        return case["rows"] * (case["window"] + case["extra"]) - half * half
    return case["rows"] * case["degree"]


def work(case):
    nnz, rows, cols, k, e = _nonzeros(case), case["rows"], case["cols"], case["k"], BYTES[case["dtype"]]
    pattern = 4 * nnz + 4 * (rows + 1)  # column indices and row offsets
    value = 8 if case["dtype"] == "f64" else 4
    heads = case.get("heads", 1)
    op = case["op"]
    if op == "build":  # the pattern once, and the lists (a row has about one entry)
        return {"bytes": pattern + 8 * rows, "flops": 0}
    if op == "sddmm":  # the sampled values are read and written
        return {"bytes": pattern + 8 * nnz + (rows + cols) * k * e, "flops": 2 * nnz * k}
    if op == "spmm":
        return {"bytes": pattern + value * nnz + cols * k * e + rows * k * value, "flops": 2 * nnz * k}
    if op == "spmm_train":  # the operand and the output, the output's gradient and the operand's
        return {"bytes": pattern + 4 * nnz + 2 * cols * k * e + 2 * rows * k * 4, "flops": 4 * nnz * k}
    if op == "attention":  # scores and weighted sum
        return {"bytes": pattern + 4 * nnz + heads * k * ((rows + 2 * cols) * e + rows * 4), "flops": 4 * nnz * k * heads}
    # the forward's two products and the backward's four (dp, dq, dk, dv)
    return {"bytes": pattern + 4 * nnz + heads * k * (2 * (rows + 2 * cols) * e + 2 * rows * 4), "flops": 12 * nnz * k * heads}


def tolerance(case):
    if case["op"] == "build":
        return "exact"
    if case["dtype"] == "f64":
        return {"rel": 1e-12}
    if case["dtype"] == "f16" and case["op"] in ("spmm_train", "attention_train"):
        return {"rel": 2e-3}  # gradients in half precision
    return {"rel": 1e-5}  # 16-bit operands are summed in 32 bits too
