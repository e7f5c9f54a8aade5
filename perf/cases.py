"""Performance cases: calls of the public ops over the sizes, element types
and options that programs give them.

Each case is one call (or, for the row ops, the four calls of an edge
softmax) on operands resident on the GPU, with the options object and the
output buffers that a program keeps between calls.  Sizes are those of the
five benchmark configurations (sparsewavecomp_amd/workloads.py) or generic;
``draw`` spreads the same calls over the ranges in ``RANGES``.

The inputs come from the seed alone and are made on the GPU.  ``exact``
recomputes a case in float64 with plain torch.
"""
import math

import torch

import sparsewavecomp_amd as sw

DEV = "cuda"

# the option strings of the README and of bench.py's tuned mappings; "" is a
# call without options (the reference's mappings)
SPMV_POSITION = ("spmv-mapping=wave-per-position spmv-positions-per-lane=4 "
                 "spmv-block-size=64")
SPMV_ROWS = "spmv-mapping=wave-per-row spmv-lanes-per-row=16"
SPMM_TILE = ("spmm-mapping=wave-per-row-tile spmm-tile-size=32 "
             "spmm-lanes-per-row=64 spmm-block-size=64")
SDDMM_WAVE = "sddmm-mapping=wave-per-row"
SDDMM_TILE = "sddmm-mapping=row-tile-mfma"
ATTENTION_FUSED = ("sddmm-mapping=row-tile-mfma sddmm-lanes-per-row=64 "
                   "spmm-mapping=row-tile-mfma")

# what draw() spreads over (log-uniform where the range passes a factor of
# ten), and the caps that keep a drawn case below the largest listed one
RANGES = {
    "rows": (1000, 1 << 20),         # CSR rows of SpMV, COO, SpMM, row ops
    "mean": (4, 64),                 # stored entries per row, lognormal
    "k": (1, 128),                   # dense columns of SpMM
    "nnz_cap": 20_000_000,
    "nnz_k_cap": 500_000_000,        # nnz * k of SpMM and SDDMM
    "bsr_block_rows": (100, 16384),
    "bsr_k": (8, 256),
    "seq": (500, 16384),
    "kdim": (16, 256),               # SDDMM dot length
}


def listed():
    return [
        # One small product inside a solver loop: configuration 1 (4096 rows
        # of exactly 16 entries), no options.  Launch and host time count.
        {"name": "spmv_small", "op": "spmv", "rows": 4096, "cols": 4096,
         "mean": 16, "sigma": 0.0, "options": ""},
        # A graph-sized product: configuration 2, 1M rows with lognormal
        # lengths up to 4096, the headline mapping.
        {"name": "spmv_power_law", "op": "spmv", "rows": 1 << 20,
         "cols": 1 << 20, "mean": 32, "sigma": 1.5, "options": SPMV_POSITION},
        # A Matrix Market matrix multiplied as it was read, as row-sorted COO
        # entries, no options; rows and columns differ and are odd.
        {"name": "coo_default", "op": "coo", "rows": 300007, "cols": 250013,
         "mean": 16, "sigma": 1.0, "options": ""},
        # Graph features: configuration 3 with 64 dense columns, the
        # row-tile mapping; the largest case.
        {"name": "spmm_f32_k64", "op": "spmm", "rows": 1 << 20,
         "cols": 1 << 20, "mean": 32, "sigma": 1.5, "k": 64, "dtype": "f32",
         "options": SPMM_TILE},
        # A bf16 feature matrix of 100 columns (no power of two), no options.
        {"name": "spmm_bf16_k100", "op": "spmm", "rows": 200003,
         "cols": 180001, "mean": 20, "sigma": 1.0, "k": 100, "dtype": "bf16",
         "options": ""},
        # A block-sparse weight matrix in fp32: configuration 4 (16 x 16
        # blocks, 8 per block row, 128 columns).
        {"name": "bsr_f32_b16", "op": "bsr", "block_rows": 16384, "b": 16,
         "blocks": 8, "keep": 1.0, "k": 128, "dtype": "f32",
         "out": "f32"},
        # A block-sparse linear layer in bf16 with 32 x 32 blocks, ragged
        # block rows, 200 columns (a partial column strip).
        {"name": "bsr_bf16_b32", "op": "bsr", "block_rows": 2048, "b": 32,
         "blocks": 12, "keep": 0.75, "k": 200, "dtype": "bf16",
         "out": "bf16"},
        # One attention head as the bundle has it: configuration 5 (8192
        # positions, 64 x 64 blocks, window 4 + 2 random, d = 64), the
        # one-kernel options.
        {"name": "attention_f32", "op": "attention", "seq": 8192, "block": 64,
         "window": 4, "random": 2, "d": 64, "dv": 64, "dtype": "f32",
         "bias": False, "options": ATTENTION_FUSED},
        # A longer bf16 head with a wider window: 16384 positions of up to
        # 768 entries each, d = 128, an additive bias on the entries.
        {"name": "attention_bf16_wide", "op": "attention", "seq": 16384,
         "block": 64, "window": 8, "random": 4, "d": 128, "dv": 128,
         "dtype": "bf16", "bias": True, "options": ATTENTION_FUSED},
        # A short head of an odd length called without options.
        {"name": "attention_default", "op": "attention", "seq": 3001,
         "block": 64, "window": 4, "random": 2, "d": 64, "dv": 64,
         "dtype": "f32", "bias": True, "options": ""},
        # Edge scores of a graph (no block structure), no options.
        {"name": "sddmm_graph", "op": "sddmm", "rows": 60013, "cols": 50021,
         "mean": 16, "sigma": 1.0, "kdim": 64, "dtype": "f32",
         "options": ""},
        # Softmax over each vertex's edges as the four row ops, no options.
        {"name": "edge_softmax", "op": "rowops", "rows": 300007, "mean": 24,
         "sigma": 1.2, "dtype": "f32", "options": ""},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["spmv", "coo", "spmm", "bsr", "attention", "sddmm",
                     "rowops"])
    dtype = rng.choice(["f32", "bf16"])
    if op == "bsr":
        b = rng.choice([8, 16, 32, 64])
        k = _log_int(rng, *RANGES["bsr_k"])
        blocks = rng.randint(3, 16)
        top = int(3.4e7 / (b * b * blocks * (k / 128)))
        return {"op": op, "b": b, "blocks": blocks, "k": k, "dtype": dtype,
                "keep": round(rng.uniform(0.5, 1.0), 2),
                "block_rows": min(_log_int(rng, *RANGES["bsr_block_rows"]),
                                  max(top, 100)),
                "out": rng.choice(["f32", "bf16"]) if dtype == "bf16"
                else "f32"}
    if op == "attention":
        seq = _log_int(rng, *RANGES["seq"])
        block = rng.choice([32, 64, 128])
        window, random_blocks = rng.randint(1, 6), rng.randint(0, 3)
        while (window + random_blocks) * block > 768:
            block //= 2
        return {"op": op, "seq": seq, "block": block,
                "window": window, "random": random_blocks,
                "d": rng.choice([32, 64, 64, 96, 128, 128]),
                "dv": rng.choice([64, 64, 80, 128]),
                "dtype": dtype, "bias": rng.random() < 0.5,
                "options": rng.choice([ATTENTION_FUSED, ATTENTION_FUSED, ""])}
    mean = rng.randint(*RANGES["mean"])
    rows = _log_int(rng, *RANGES["rows"])
    case = {"op": op, "mean": mean, "sigma": round(rng.uniform(0.0, 1.5), 2),
            "options": ""}
    width = 1
    if op == "spmm":
        case["k"] = width = _log_int(rng, *RANGES["k"])
        case["options"] = rng.choice(["", SPMM_TILE])
    elif op == "sddmm":
        case["kdim"] = width = _log_int(rng, *RANGES["kdim"])
        case["options"] = rng.choice(["", SDDMM_WAVE, SDDMM_TILE])
        width *= 4  # a gather per term
    elif op == "spmv":
        case["options"] = rng.choice(["", SPMV_ROWS, SPMV_POSITION])
    elif op == "coo":
        case["options"] = rng.choice(["", SPMV_POSITION])
    if op in ("spmm", "sddmm", "rowops"):
        case["dtype"] = dtype
    cap = min(RANGES["nnz_cap"], RANGES["nnz_k_cap"] // width)
    case["rows"] = max(min(rows, cap // mean), 500)
    if op != "rowops":
        case["cols"] = max(500, int(case["rows"] * rng.uniform(0.5, 1.5)))
    return case


# ---- inputs -----------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _torch_dtype(name):
    return torch.float32 if name == "f32" else torch.bfloat16


def _uniform(g, *shape):
    return torch.rand(shape, generator=g, device=DEV) * 2.0 - 1.0


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _csr(g, rows, cols, mean, sigma):
    """(row offsets, columns): lognormal row lengths clipped to [1, 4096],
    distinct sorted uniform columns (sort(u_i) + i)."""
    top = min(4096, cols)
    lengths = torch.full((rows,), float(mean), device=DEV)
    if sigma > 0:  # the lognormal's quantiles in a random row order
        at = (torch.arange(rows, device=DEV, dtype=torch.float64) + 0.5) / rows
        normal = math.sqrt(2.0) * torch.erfinv(2.0 * at - 1.0)
        lengths = torch.exp(math.log(mean) - sigma * sigma / 2.0
                            + sigma * normal)
        lengths = lengths[torch.randperm(rows, generator=g, device=DEV)]
    lengths = lengths.round().clamp(1, top).long()
    ro = torch.zeros(rows + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(lengths, 0, out=ro[1:])
    row = torch.repeat_interleave(lengths)
    span = cols - lengths + 1
    u = (torch.rand(row.numel(), generator=g, device=DEV,
                    dtype=torch.float64) * span[row]).long()
    u = torch.minimum(u, span[row] - 1)
    key = (row * cols + u).sort().values - row * cols
    col = key + torch.arange(row.numel(), device=DEV) - ro[row]
    return ro.int(), col.int()


def _bsr(g, block_rows, blocks, keep):
    """(block row offsets, block columns): the diagonal, half of the blocks
    at distinct offsets within +-4 of it, the rest anywhere; a block off the
    diagonal stays with probability keep."""
    i = torch.arange(block_rows, device=DEV)
    near = torch.rand((block_rows, 8), generator=g,
                      device=DEV).topk(blocks // 2, 1).indices - 4
    near = i[:, None] + torch.where(near >= 0, near + 1, near)
    far = torch.randint(0, block_rows, (block_rows, blocks - blocks // 2 - 1),
                        generator=g, device=DEV)
    other = torch.cat([near, far], 1)
    stays = torch.rand(other.shape, generator=g, device=DEV) < keep
    stays &= (other >= 0) & (other < block_rows)
    key = torch.where(stays, other, i[:, None]) + i[:, None] * block_rows
    key = torch.unique(torch.cat([i * (block_rows + 1), key.reshape(-1)]))
    bro = torch.zeros(block_rows + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(torch.bincount(key // block_rows, minlength=block_rows), 0,
                 out=bro[1:])
    return bro.int(), (key % block_rows).int()


def _mask(g, seq, block, window, random_blocks):
    """(row offsets, columns) of a causal block mask: a window of blocks
    ending at the diagonal and random blocks before it, the last block of
    the sequence partial where block does not divide it."""
    nb = -(-seq // block)
    b = torch.arange(nb, device=DEV)
    first = (b - window + 1).clamp(min=0)
    take = min(random_blocks, nb)
    score = torch.rand((nb, nb), generator=g, device=DEV)
    score = score.masked_fill(b[None, :] >= first[:, None], -1.0)
    top = score.topk(take, 1) if take else None
    lists = [b[:, None] - torch.arange(window, device=DEV)]
    if take:
        lists.append(torch.where(top.values >= 0, top.indices, -1))
    blocks = torch.cat(lists, 1)
    blocks = torch.where(blocks < 0, nb, blocks).sort(1).values
    count = (blocks < nb).sum(1)
    r = torch.arange(seq, device=DEV)
    rb = r // block
    lengths = (count[rb] - 1) * block + r % block + 1
    ro = torch.zeros(seq + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(lengths, 0, out=ro[1:])
    row = torch.repeat_interleave(lengths)
    t = torch.arange(row.numel(), device=DEV) - ro[row]
    col = blocks[rb[row], t // block] * block + t % block
    return ro.int(), col.int()


def prepare(case, seed):
    g = _gen(seed)
    op = case["op"]
    text = case.get("options", "")
    s = {"op": op, "options": sw.Options.parse(text) if text else None}
    dt = _torch_dtype(case.get("dtype", "f32"))
    if op == "bsr":
        b, k = case["b"], case["k"]
        s["b"] = b
        s["ro"], s["col"] = _bsr(g, case["block_rows"], case["blocks"],
                                 case["keep"])
        n = case["block_rows"] * b
        s["val"] = (0.02 * _normal(g, s["col"].numel(), b, b)).to(dt)
        s["rhs"] = _normal(g, n, k).to(dt)
        s["out"] = torch.empty((n, k), device=DEV,
                               dtype=_torch_dtype(case["out"]))
        return s
    if op == "attention":
        seq, d, dv = case["seq"], case["d"], case["dv"]
        s["ro"], s["col"] = _mask(g, seq, case["block"], case["window"],
                                  case["random"])
        nnz = s["col"].numel()
        bias = (_normal(g, nnz) if case["bias"]
                else torch.zeros(nnz, device=DEV))
        s["mask"] = bias.to(dt)
        s["beta"] = 1.0 if case["bias"] else 0.0
        s["alpha"] = 1.0 / math.sqrt(d)
        s["q"] = _normal(g, seq, d).to(dt)
        s["kt"] = _normal(g, seq, d).to(dt).t().contiguous()
        s["v"] = _normal(g, seq, dv).to(dt)
        s["scores"] = torch.empty(nnz, device=DEV, dtype=dt)
        s["rmax"] = torch.empty(seq, device=DEV, dtype=dt)
        s["rsum"] = torch.empty(seq, device=DEV, dtype=dt)
        s["out"] = torch.empty((seq, dv), device=DEV, dtype=dt)
        return s
    rows, cols = case["rows"], case.get("cols", case["rows"])
    s["ro"], s["col"] = _csr(g, rows, cols, case["mean"], case["sigma"])
    nnz = s["col"].numel()
    if op == "rowops":
        s["val"] = (2.0 * _normal(g, nnz)).to(dt)
        s["rmax"] = torch.empty(rows, device=DEV, dtype=dt)
        s["rsum"] = torch.empty(rows, device=DEV, dtype=dt)
        s["exps"] = torch.empty(nnz, device=DEV, dtype=dt)
        s["out"] = torch.empty(nnz, device=DEV, dtype=dt)
        return s
    s["val"] = _uniform(g, nnz).to(dt)
    if op == "sddmm":
        s["lhs"] = _normal(g, rows, case["kdim"]).to(dt)
        s["rhs"] = _normal(g, case["kdim"], cols).to(dt)
        s["out"] = torch.empty(nnz, device=DEV, dtype=dt)
    elif op == "spmm":
        s["rhs"] = _uniform(g, cols, case["k"]).to(dt)
        s["out"] = torch.empty((rows, case["k"]), device=DEV, dtype=dt)
    else:
        s["x"] = _uniform(g, cols)
        s["out"] = torch.empty(rows, device=DEV)
        if op == "coo":
            s["ri"] = _rows(s["ro"]).int()
    return s


def run(s):
    op, o = s["op"], s["options"]
    if op == "spmv":
        return sw.spmv(s["ro"], s["col"], s["val"], s["x"], s["out"],
                       options=o)
    if op == "coo":
        return sw.coo_spmv(s["ri"], s["col"], s["val"], s["x"], s["out"],
                           options=o)
    if op == "spmm":
        return sw.spmm(s["ro"], s["col"], s["val"], s["rhs"], s["out"],
                       options=o)
    if op == "bsr":
        return sw.bsr_spmm(s["ro"], s["col"], s["val"], s["rhs"], s["out"],
                           s["b"], options=o)
    if op == "attention":
        sw.sparse_attention(s["ro"], s["col"], s["mask"], s["q"], s["kt"],
                            s["v"], s["scores"], s["rmax"], s["rsum"],
                            s["out"], s["alpha"], s["beta"], options=o)
        return {"scores": s["scores"], "rmax": s["rmax"], "rsum": s["rsum"],
                "out": s["out"]}
    if op == "sddmm":
        return sw.sddmm(s["ro"], s["col"], s["val"], s["lhs"], s["rhs"],
                        s["out"], sw.SDDMM_MUL, options=o)
    sw.csr_row_reduce(s["ro"], s["col"], s["val"], s["rmax"], "max",
                      options=o)
    sw.csr_rowwise_map(s["ro"], s["col"], s["val"], s["rmax"], s["exps"],
                       sw.MAP_EXP_SUB, options=o)
    sw.csr_row_reduce(s["ro"], s["col"], s["exps"], s["rsum"], "sum",
                      options=o)
    sw.csr_rowwise_map(s["ro"], s["col"], s["exps"], s["rsum"], s["out"],
                       sw.MAP_DIV, options=o)
    return {"rmax": s["rmax"], "exps": s["exps"], "rsum": s["rsum"],
            "out": s["out"]}


# ---- what a pass cannot do without ------------------------------------------

def work(case):
    op = case["op"]
    e = 4 if case.get("dtype", "f32") == "f32" else 2
    if op == "bsr":
        b, k, br = case["b"], case["k"], case["block_rows"]
        nnzb = br * (1 + (case["blocks"] - 1) * case["keep"])
        eo = 4 if case["out"] == "f32" else 2
        return {"bytes": 4 * (br + 1) + 4 * nnzb + e * nnzb * b * b
                + (e + eo) * br * b * k,
                "flops": 2 * nnzb * b * b * k}
    if op == "attention":
        seq, d, dv = case["seq"], case["d"], case["dv"]
        row = (case["window"] + case["random"] - 0.5) * case["block"]
        nnz = seq * min(row, seq / 2)
        return {"bytes": 4 * (seq + 1) + (4 + 2 * e) * nnz
                + e * seq * (2 * d + 2 * dv + 2),
                "flops": nnz * (2 * d + 2 * dv + 6)}
    rows = case["rows"]
    nnz = rows * case["mean"]  # expected; clipping moves it little
    if op == "rowops":
        # max, exp, sum, divide: four calls, each reading its operands and
        # writing its result once
        return {"bytes": 4 * 4 * (rows + 1) + e * (4 * rows + 6 * nnz),
                "flops": 5 * nnz}
    cols = case["cols"]
    if op == "spmv":
        return {"bytes": 4 * (rows + 1) + 8 * nnz + 4 * (rows + cols),
                "flops": 2 * nnz}
    if op == "coo":
        return {"bytes": 12 * nnz + 4 * (rows + cols), "flops": 2 * nnz}
    if op == "spmm":
        k = case["k"]
        return {"bytes": 4 * (rows + 1) + (4 + e) * nnz
                + e * k * (rows + cols), "flops": 2 * nnz * k}
    k = case["kdim"]
    return {"bytes": 4 * (rows + 1) + (4 + 2 * e) * nnz
            + e * k * (rows + cols), "flops": 2 * nnz * k}


def tolerance(case):
    """fp32: sums of tens to thousands of fp32 terms in any order stay within
    a few 1e-7 of the exact sum in the 2-norm.  bf16: each stored value is
    rounded once (2^-9), and the attention chain rounds its scores, so a
    probability moves with the rounding of scores of a few units."""
    if case.get("dtype", "f32") == "f32":
        return {"rel": 4e-6, "max": 1e-4}
    if case["op"] == "attention":
        return {"rel": 2e-2, "max": 0.2}
    return {"rel": 8e-3, "max": 2e-2}


# ---- float64 recomputation --------------------------------------------------

def _rows(ro):
    return torch.repeat_interleave((ro[1:] - ro[:-1]).long())


def _row_sums(row, values, rows):
    out = torch.zeros((rows,) + values.shape[1:], dtype=torch.float64,
                      device=DEV)
    return out.index_add_(0, row, values)


def _chunks(nnz, width):
    step = max(1, (1 << 27) // width)
    return [(a, min(a + step, nnz)) for a in range(0, nnz, step)]


def _dots(row, col, lhs, rhs_t):
    """lhs[row] . rhs_t[col] per entry, in float64."""
    out = torch.empty(row.numel(), dtype=torch.float64, device=DEV)
    for a, z in _chunks(row.numel(), lhs.shape[1]):
        out[a:z] = (lhs[row[a:z]] * rhs_t[col[a:z]]).sum(1)
    return out


def _products(row, col, val, rhs, rows):
    """sum of val * rhs[col] over each row's entries, in float64."""
    out = torch.zeros((rows, rhs.shape[1]), dtype=torch.float64, device=DEV)
    for a, z in _chunks(row.numel(), rhs.shape[1]):
        out.index_add_(0, row[a:z], val[a:z, None] * rhs[col[a:z]])
    return out


def _softmax_parts(row, x, rows):
    rmax = torch.full((rows,), -math.inf, dtype=torch.float64, device=DEV)
    rmax.scatter_reduce_(0, row, x, "amax")
    exps = torch.exp(x - rmax[row])
    rsum = _row_sums(row, exps, rows)
    return rmax, exps, rsum, exps / rsum[row]


def exact(case, seed):
    s = prepare(case, seed)
    op = case["op"]
    col = s["col"].long()
    if op == "bsr":
        b, k = case["b"], case["k"]
        brow = _rows(s["ro"])
        rhs = s["rhs"].double().reshape(-1, b, k)
        out = torch.zeros_like(rhs)
        for a, z in _chunks(col.numel(), b * max(b, k)):
            out.index_add_(0, brow[a:z], torch.bmm(s["val"][a:z].double(),
                                                   rhs[col[a:z]]))
        return out.reshape(-1, k)
    row = _rows(s["ro"])
    if op == "attention":
        seq = case["seq"]
        x = (s["alpha"] * _dots(row, col, s["q"].double(),
                                s["kt"].double().t().contiguous())
             + s["beta"] * s["mask"].double())
        rmax, _, rsum, p = _softmax_parts(row, x, seq)
        return {"scores": p, "rmax": rmax, "rsum": rsum,
                "out": _products(row, col, p, s["v"].double(), seq)}
    rows = case["rows"]
    val = s["val"].double()
    if op == "rowops":
        rmax, exps, rsum, p = _softmax_parts(row, val, rows)
        return {"rmax": rmax, "exps": exps, "rsum": rsum, "out": p}
    if op == "sddmm":
        return val * _dots(row, col, s["lhs"].double(),
                           s["rhs"].double().t().contiguous())
    if op == "spmm":
        return _products(row, col, val, s["rhs"].double(), rows)
    return _row_sums(row, val * s["x"].double()[col], rows)
